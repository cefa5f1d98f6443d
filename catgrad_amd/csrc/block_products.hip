// Products of operands that lie narrow in memory (bfloat16, binary16 or fp8 patterns, k contiguous) with the sums in 32 bits, for
// shapes that do not fill the device with 256 x 256 tiles: y[M, N] = x[M, K] . w[N, K]^T, cut along k as well when there are few
// tiles.  The result is 32-bit words, or rounded to the operands' format in the last store.
#include "blocks.hpp"
#include "gemm_args.hpp"

#include <algorithm>
#include <cmath>

namespace cg {
namespace {

constexpr int kThreads = 256;
constexpr uint32_t kTileN = 128, kStages = 4, kStageBytes = 64, kXcds = 8, kGroupM = 8;
typedef float float16v __attribute__((ext_vector_type(16)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef int int4v __attribute__((ext_vector_type(4)));

struct TileArgs {
    const char *x, *w;
    void *y;                   // split s of y at y + s * M * N
    uint32_t M, N, ld;         // ld: elements from row to row of y
    uint32_t K;                // bytes, as the pitches
    uint32_t x_pitch, w_pitch;
    uint32_t k_part;           // bytes of k per split, a multiple of kStageBytes
};

template <int FMT> __device__ __forceinline__ uint32_t pattern(float v) {
    if constexpr (FMT == kFmtBF16) return round_bf16_bits(asu(v)) >> 16;
    else if constexpr (FMT == kFmtF16) return __half_as_ushort(__float2half_rn(v));
    else {
        // (the rounding pass's byte in one conversion: magnitudes clamped to the largest, NaNs set apart)
        const uint32_t u = asu(v), m = u & 0x7FFFFFFFu, sign = u & 0x80000000u;
        const float c = asf(min(m, 0x43E00000u) | sign);
        return m > 0x7F800000u ? sign >> 24 | 0x7Fu : (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(c, c, 0, false) & 0xFFu;
    }
}
template <int FMT> __device__ __forceinline__ void put(void *y, uint64_t at, float v) {
    if constexpr (FMT == kFmtWords) static_cast<float *>(y)[at] = v;
    else if constexpr (FMT == kFmtF8) static_cast<uint8_t *>(y)[at] = (uint8_t)pattern<FMT>(v);
    else static_cast<uint16_t *>(y)[at] = (uint16_t)pattern<FMT>(v);
}

__device__ const uint32_t kZeros[4] __attribute__((aligned(16))) = {0, 0, 0, 0};

// 64 MT x 128 tiles, four waves of 32 MT x 64 each.  A stage is 64 bytes of k per row, fetched by loads straight into LDS in
// a ring of four: one multiplied, three in flight, one barrier a stage.  A row's four 16-byte columns lie at column
// c ^ ((row >> 2) & 3), so that the lanes that a 128-bit read serves together cover all banks; a load instruction of a wave
// fills 16 rows in lane order.  Rows beyond the edge are clamped, columns beyond K come from a block of zeros.  FMT: the operands'
// format; OUT: the result's.
template <int FMT, int OUT, int MT> __global__ __launch_bounds__(kThreads) void narrow_tile_kernel(const TileArgs a) {
    constexpr uint32_t TM = 64 * MT, A_BYTES = TM * 64, STAGE = A_BYTES + kTileN * 64;
    extern __shared__ float lds_dyn[];
    typedef __attribute__((address_space(3))) char lds_char;
    lds_char *const lds = (lds_char *)lds_dyn;

    // a run of tiles per XCD, down a column of kGroupM row tiles first
    const uint32_t tiles_n = (a.N + kTileN - 1) / kTileN, tiles_m = (a.M + TM - 1) / TM, ntiles = tiles_m * tiles_n;
    const uint32_t xcd = blockIdx.x % kXcds, q8 = ntiles / kXcds, r8 = ntiles % kXcds;
    const uint32_t lin = xcd * q8 + min(xcd, r8) + blockIdx.x / kXcds;
    const uint32_t group = lin / (kGroupM * tiles_n), in_group = lin % (kGroupM * tiles_n), first_m = group * kGroupM;
    const uint32_t gsize = min(tiles_m - first_m, kGroupM);
    const uint32_t m0 = (first_m + in_group % gsize) * TM, n0 = (in_group / gsize) * kTileN;
    const uint32_t k_first = blockIdx.y * a.k_part, k_end = min(k_first + a.k_part, a.K), nk = (k_end - k_first + kStageBytes - 1) / kStageBytes;

    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64;
    const uint32_t wm = (wave / 2) * 32 * MT, wn = (wave % 2) * 64, li = lane % 32, lg = lane / 32;

    // this lane's part of the wave's loads of a stage: MT of x, two of w; `col`: the logical 16-byte column it fetches
    uint32_t off[MT + 2];
    const uint32_t col = (lane % 4) ^ ((lane >> 4) & 3); // ((row >> 2) & 3 with row = 16 n + lane / 4)
#pragma unroll
    for (int q = 0; q < MT; q++) off[q] = min(m0 + (wave * MT + q) * 16 + lane / 4, a.M - 1) * a.x_pitch + col * 16;
#pragma unroll
    for (int q = 0; q < 2; q++) off[MT + q] = min(n0 + (wave * 2 + q) * 16 + lane / 4, a.N - 1) * a.w_pitch + col * 16;
    auto issue = [&](const uint32_t stage, const uint32_t place) {
        const uint32_t k0 = k_first + stage * kStageBytes;
        const bool tail = k0 + kStageBytes > a.K, outside = k0 + col * 16 >= a.K;
#pragma unroll
        for (int q = 0; q < MT + 2; q++) {
            const char *p = (q < MT ? a.x : a.w) + k0 + off[q];
            if (tail && outside) p = reinterpret_cast<const char *>(kZeros);
            lds_char *const l = lds + place * STAGE + (q < MT ? (wave * MT + q) * 1024 : A_BYTES + (wave * 2 + q - MT) * 1024);
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)p, (__attribute__((address_space(3))) void *)l, 16, 0, 0);
        }
    };
    const uint32_t sw = (li >> 2) & 3;
    auto frag = [&](const uint32_t base, const uint32_t c) {
        return *reinterpret_cast<const __attribute__((address_space(3))) int4v *>(lds + base + li * 64 + ((c ^ sw) * 16));
    };

    float16v acc[MT][2];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[i][j][v] = 0.0f;

    // (behind the last stage the last one is asked for again: one count of loads in flight, and a place that nobody reads)
    for (uint32_t s = 0; s < kStages - 1; s++) issue(min(s, nk - 1), s);
    for (uint32_t kt = 0; kt < nk; kt++) {
        constexpr uint32_t n = 2 * (MT + 2); // two younger stages may be in flight
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0x0070 | n); // vmcnt(n) lgkmcnt(0)
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        issue(min(kt + kStages - 1, nk - 1), (kt + kStages - 1) % kStages);
        const uint32_t base = (kt % kStages) * STAGE;
#pragma unroll
        for (int c = 0; c < 2; c++) {
            constexpr int STEPS = FMT == kFmtF8 ? 2 : 1; // matrix instructions per 16-byte column
            int4v fa[MT][STEPS], fb[2][STEPS];
            auto read = [&](const uint32_t at, int4v(&f)[STEPS]) {
                const int4v v = frag(at, c * 2 + lg);
                if constexpr (FMT != kFmtF8) f[0] = v;
                else {
                    // fp8 values are bfloat16 values: the fp8 instructions keep 3.5e-6 of a sum (64 and 2048 values of k alike),
                    // the bfloat16 ones all of its 32 bits
#pragma unroll
                    for (int w = 0; w < 4; w++) {
                        f[w / 2][w % 2 * 2] = __builtin_bit_cast(int, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8((uint32_t)v[w], 1.0f, false));
                        f[w / 2][w % 2 * 2 + 1] = __builtin_bit_cast(int, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8((uint32_t)v[w], 1.0f, true));
                    }
                }
            };
#pragma unroll
            for (int i = 0; i < MT; i++) read(base + (wm + i * 32) * 64, fa[i]);
#pragma unroll
            for (int j = 0; j < 2; j++) read(base + A_BYTES + (wn + j * 32) * 64, fb[j]);
#pragma unroll
            for (int t = 0; t < STEPS; t++)
#pragma unroll
                for (int i = 0; i < MT; i++)
#pragma unroll
                    for (int j = 0; j < 2; j++) {
                        if constexpr (FMT == kFmtF16)
                            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, fa[i][t]), __builtin_bit_cast(f16x8, fb[j][t]), acc[i][j], 0, 0, 0);
                        else
                            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, fa[i][t]), __builtin_bit_cast(bf16x8, fb[j][t]), acc[i][j], 0, 0, 0);
                    }
        }
    }
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0070); // no load may write LDS that another workgroup gets

    const uint64_t first = (uint64_t)blockIdx.y * a.M * a.N;
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const uint32_t n = n0 + wn + j * 32 + li;
            if (n >= a.N) continue;
#pragma unroll
            for (int v = 0; v < 16; v++) { // the instruction's result: row 8 (v / 4) + 4 lg + v % 4, column li
                const uint32_t m = m0 + wm + i * 32 + 8 * (v / 4) + 4 * lg + (v % 4);
                if (m < a.M) put<OUT>(a.y, first + (uint64_t)m * a.ld + n, acc[i][j][v]);
            }
        }
}

// y[e] = the parts' sum, in their order; row4 and ld4: fours of columns in a row of the parts, and from row to row of y
template <int OUT> __global__ __launch_bounds__(kThreads) void sum_parts_kernel(const float4v *part, void *y, uint32_t parts, uint64_t n4, uint32_t row4, uint32_t ld4) {
    uint64_t i = (uint64_t)blockIdx.x * kThreads + threadIdx.x;
    if (i >= n4) return;
    float4v v = __builtin_nontemporal_load(part + i);
    for (uint32_t s = 1; s < parts; s++) v += __builtin_nontemporal_load(part + s * n4 + i);
    if (row4 != ld4) i = i / row4 * ld4 + i % row4;
    if constexpr (OUT == kFmtWords) static_cast<float4v *>(y)[i] = v;
    else if constexpr (OUT == kFmtF8)
        static_cast<uint32_t *>(y)[i] = pattern<OUT>(v[0]) | pattern<OUT>(v[1]) << 8 | pattern<OUT>(v[2]) << 16 | pattern<OUT>(v[3]) << 24;
    else static_cast<uint2 *>(y)[i] = make_uint2(pattern<OUT>(v[0]) | pattern<OUT>(v[1]) << 16, pattern<OUT>(v[2]) | pattern<OUT>(v[3]) << 16);
}

// A few dozen rows: 16 RT x 16 results per workgroup, whose waves take turns of 128 bytes of k.  The operands go from memory into the
// matrix instruction's registers as they lie (16 bytes of a row per lane, four lanes side by side), two turns in flight, and the
// waves' sums meet in LDS, so that k is cut eight ways without a second launch.  WHOLE: k is whole turns.
// Bound by latency, as the tiles are at such sizes, but with one trip behind the other instead of a stage behind the other; tiles with
// the launch that adds their parts, and here, in us: bf16 32 x 576 x 576 7.8 and 3.5, 64 x 1024 x 1024 9.2 and 4.4, 128 x 3072 x 1024
// 13.5 and 10.9, 1500 x 16 x 2048 11.1 and 5.9; fp8 64 x 2048 x 2048 10.4 and 5.6.  Four row blocks: within 10 % of the better of one
// and two where they were the fastest at all.
constexpr int kThinWaves = 8, kTurnBytes = 128;
template <int FMT, int OUT, int RT, bool WHOLE> __global__ __launch_bounds__(64 * kThinWaves) void narrow_thin_kernel(const TileArgs a) {
    constexpr uint32_t TILE = RT * 256;
    __shared__ float red[kThinWaves][TILE];
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64, li = lane % 16, lg = lane / 16;
    const uint32_t n0 = blockIdx.x * 16, m0 = blockIdx.y * (16 * RT), turns = (a.K + kTurnBytes - 1) / kTurnBytes;
    const char *const col = a.w + (uint64_t)min(n0 + li, a.N - 1) * a.w_pitch, *row[RT];
#pragma unroll
    for (int i = 0; i < RT; i++) row[i] = a.x + (uint64_t)min(m0 + 16 * i + li, a.M - 1) * a.x_pitch; // (rows behind the last repeat it)
    int4v x[2][RT][2], y[2][2];
    auto ask = [&](const uint32_t t, const int set) {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const uint32_t k0 = t * kTurnBytes + h * 64 + lg * 16, k = WHOLE ? k0 : min(k0, a.K - 16);
            y[set][h] = *reinterpret_cast<const int4v *>(col + k);
#pragma unroll
            for (int i = 0; i < RT; i++) x[set][i][h] = *reinterpret_cast<const int4v *>(row[i] + k);
        }
    };
    float4v acc[RT];
#pragma unroll
    for (int i = 0; i < RT; i++) acc[i] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
    constexpr int STEPS = FMT == kFmtF8 ? 2 : 1; // matrix instructions per 16 bytes
    auto widen = [&](const int4v v, const bool in, int4v(&f)[STEPS]) { // (what was read elsewhere becomes zeros)
        if constexpr (FMT != kFmtF8) f[0] = v;
        else {
#pragma unroll
            for (int w = 0; w < 4; w++) { // (as bfloat16: see narrow_tile_kernel)
                f[w / 2][w % 2 * 2] = __builtin_bit_cast(int, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8((uint32_t)v[w], 1.0f, false));
                f[w / 2][w % 2 * 2 + 1] = __builtin_bit_cast(int, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8((uint32_t)v[w], 1.0f, true));
            }
        }
        if (WHOLE) return;
#pragma unroll
        for (int t = 0; t < STEPS; t++)
#pragma unroll
            for (int j = 0; j < 4; j++) f[t][j] = in ? f[t][j] : 0;
    };
    auto multiply = [&](const uint32_t t, const int set) {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const bool in = t * kTurnBytes + h * 64 + lg * 16 < a.K;
            int4v p[STEPS], q[STEPS];
            widen(y[set][h], in, q);
#pragma unroll
            for (int i = 0; i < RT; i++) {
                widen(x[set][i][h], in, p);
#pragma unroll
                for (int s = 0; s < STEPS; s++) {
                    if constexpr (FMT == kFmtF16) acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, p[s]), __builtin_bit_cast(f16x8, q[s]), acc[i], 0, 0, 0);
                    else acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, p[s]), __builtin_bit_cast(bf16x8, q[s]), acc[i], 0, 0, 0);
                }
            }
        }
    };
    if (wave < turns) { // (the loads stay where they stand, and every wait in the loop knows what else is on its way)
        const uint32_t n = (turns - 1 - wave) / kThinWaves + 1;
        uint32_t t = wave;
        ask(t, 0);
        if (n == 1) {
            multiply(t, 0);
        } else {
            ask(t + kThinWaves, 1);
            for (uint32_t left = n; left > 3; left -= 2, t += 2 * kThinWaves) {
                multiply(t, 0);
                __builtin_amdgcn_sched_barrier(0);
                ask(t + 2 * kThinWaves, 0);
                __builtin_amdgcn_sched_barrier(0);
                multiply(t + kThinWaves, 1);
                __builtin_amdgcn_sched_barrier(0);
                ask(t + 3 * kThinWaves, 1);
                __builtin_amdgcn_sched_barrier(0);
            }
            multiply(t, 0);
            if (n % 2) {
                ask(t + 2 * kThinWaves, 0);
                multiply(t + kThinWaves, 1);
                multiply(t + 2 * kThinWaves, 0);
            } else {
                multiply(t + kThinWaves, 1);
            }
        }
    }
    // (the last sums are on their way behind a branch, where the compiler does not always wait for them)
#pragma unroll
    for (int i = 0; i < RT; i++) asm volatile("s_nop 7" : "+v"(acc[i]));
#pragma unroll
    for (int i = 0; i < RT; i++)
#pragma unroll
        for (int v = 0; v < 4; v++) red[wave][i * 256 + v * 64 + lane] = acc[i][v];
    __syncthreads();
    for (uint32_t e = threadIdx.x; e < TILE; e += 64 * kThinWaves) {
        float s = red[0][e];
#pragma unroll
        for (int w = 1; w < kThinWaves; w++) s += red[w][e];
        const uint32_t l = e % 64, r = m0 + e / 256 * 16 + l / 16 * 4 + e / 64 % 4, c = n0 + l % 16;
        if (r < a.M && c < a.N) put<OUT>(a.y, (uint64_t)r * a.ld + c, s);
    }
}

template <int FMT, int OUT, int RT> void launch_thin(cg_backend *be, const TileArgs &a) {
    const dim3 grid((a.N + 15) / 16, (a.M + 16 * RT - 1) / (16 * RT));
    if (a.K % kTurnBytes == 0) launch_kernel((narrow_thin_kernel<FMT, OUT, RT, true>), grid, dim3(64 * kThinWaves), 0, be->stream, a);
    else launch_kernel((narrow_thin_kernel<FMT, OUT, RT, false>), grid, dim3(64 * kThinWaves), 0, be->stream, a);
}

int launched(const char *what) {
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? CG_OK : hip_fail(e, what);
}

template <int FMT, int OUT> int run_tiles(cg_backend *be, TileArgs a) {
    const bool low = a.M <= 64;
    const uint32_t tm = low ? 64 : 128;
    const uint64_t tiles = (uint64_t)((a.M + tm - 1) / tm) * ((a.N + kTileN - 1) / kTileN);
    if (tiles > 0x7FFFFFFFull) return kDeclined;
    // Cut along k by what the launch takes (start and end, stages, parts to be written and summed), into at most two workgroups per
    // compute unit with at least 256 bytes of k each; fitted to 251 shapes of 9 to 4096 rows, every cut timed: 1 % above the fastest in
    // the mean.  As many workgroups as there is room for: 7 % above it (bf16, us: 1500 x 576 x 1536 11.8 uncut, 20.8 in two parts;
    // 2048 x 1024 x 1024 15.9 and 19.9; 64 x 2048 x 8192 12.5 in four parts, 15.6 in eight).  The same shape always gets the same cut.
    const uint64_t mn = (uint64_t)a.M * a.N, room = 2 * (uint64_t)be->compute_units;
    const bool f8 = FMT == kFmtF8;
    const double start = low ? (f8 ? 4.2 : 6.1) : f8 ? 5.4 : 6.8, stage = low ? (f8 ? 0.31 : 0.114) : f8 ? 0.58 : 0.236, share = low ? (f8 ? 0.83 : 1.0) : f8 ? 0.68 : 0.765;
    uint32_t splits = 1;
    double best = 0;
    const bool fours = mn % 4 == 0 && (a.ld == a.N || (a.N % 4 == 0 && a.ld % 4 == 0));
    for (uint32_t p = 1; p == 1 || (fours && p <= 16 && p * tiles <= room && a.K / p >= 256); p++) {
        const double rounds = std::ceil((double)(tiles * p) / be->compute_units), stages = ((a.K + p - 1) / p + kStageBytes - 1) / kStageBytes;
        const double us = start + stage * stages * std::max(1.0, share * rounds) + (p > 1 ? 0.9 + 0.15 * p + 1.44e-6 * p * mn : 0.0);
        if (p == 1 || us < best) splits = p, best = us;
    }
    // Few rows, or little work: without a second launch, where that is faster by a tenth.  Fitted to 136 shapes of 9 to 1500 rows, each
    // format and both heights timed, most within a tenth: one row block while a compute unit has one workgroup, two beyond.  The tenth errs on the
    // tiles' side: over 70 drawn shapes of 9 to 400 rows a format, what is taken is 13 % above the faster way for bf16 and 3 % for fp8 in the mean;
    // without it 9 and 0 (106 x 6224 x 100 10.3 us here and 17.6 on the tiles, estimated as even).  The f32 rule (split_gemm.hip), without one, is
    // 4 % above, 8 with it.
    int high = 0;
    best *= 0.9;
    for (int rt = 1; rt <= 2; rt++) {
        const uint64_t rows = (a.M + 16 * rt - 1) / (16 * rt);
        const double rounds = (double)(rows * ((a.N + 15) / 16)) / be->compute_units, turns = a.K / (double)(kThinWaves * kTurnBytes);
        const double us = 2.6 + (rt == 1 ? 0.9 : 1.32) * std::max(0.5, turns) * std::max(1.0, rounds);
        if (rows <= 65535 && us < best) high = rt, best = us;
    }
    if (high) {
        if (high == 1) launch_thin<FMT, OUT, 1>(be, a);
        else launch_thin<FMT, OUT, 2>(be, a);
        return launched("narrow_thin");
    }
    a.k_part = ((a.K + splits - 1) / splits + kStageBytes - 1) / kStageBytes * kStageBytes;
    splits = (a.K + a.k_part - 1) / a.k_part;
    void *parts = nullptr, *const y = a.y;
    size_t cls = 0;
    if (splits > 1 && be->pool.alloc(mn * splits * 4, &parts, &cls)) {
        (void)hipGetLastError();
        splits = 1; // no room for the parts: uncut
        a.k_part = (a.K + kStageBytes - 1) / kStageBytes * kStageBytes;
    }
    const uint32_t ld = a.ld;
    if (splits > 1) a.y = parts, a.ld = a.N;
    const dim3 grid((uint32_t)tiles, splits);
    const size_t lds = (size_t)kStages * (tm + kTileN) * kStageBytes;
    if (splits > 1) {
        if (low) launch_kernel((narrow_tile_kernel<FMT, kFmtWords, 1>), grid, dim3(kThreads), lds, be->stream, a);
        else launch_kernel((narrow_tile_kernel<FMT, kFmtWords, 2>), grid, dim3(kThreads), lds, be->stream, a);
        launch_kernel((sum_parts_kernel<OUT>), dim3((uint32_t)((mn / 4 + kThreads - 1) / kThreads)), dim3(kThreads), 0, be->stream,
                           static_cast<const float4v *>(parts), y, splits, mn / 4, a.N / 4, ld == a.N ? a.N / 4 : ld / 4);
        be->pool.free(parts, cls); // stream-ordered
    } else {
        if (low) launch_kernel((narrow_tile_kernel<FMT, OUT, 1>), grid, dim3(kThreads), lds, be->stream, a);
        else launch_kernel((narrow_tile_kernel<FMT, OUT, 2>), grid, dim3(kThreads), lds, be->stream, a);
    }
    return launched("narrow_tiles");
}

} // namespace

int launch_narrow_tiles(cg_backend *be, int fmt, const void *x, int64_t x_pitch, int64_t rows, const void *w, int64_t w_pitch, int64_t n, int64_t k, void *y, int y_fmt,
                        int64_t y_pitch) {
    const int64_t eb = (int64_t)fmt_bytes(fmt);
    if (fmt == kFmtWords || !fits_narrow_tiles(fmt, x_pitch, rows, w_pitch, n, k)) return kDeclined;
    if (y_pitch != 0 && (y_pitch < n || y_pitch >= (1ll << 31))) return kDeclined;
    if (!x || !w || reinterpret_cast<uintptr_t>(x) % 16 || reinterpret_cast<uintptr_t>(w) % 16) return kDeclined;
    TileArgs a{};
    a.x = static_cast<const char *>(x);
    a.w = static_cast<const char *>(w);
    a.y = y;
    a.M = (uint32_t)rows;
    a.N = (uint32_t)n;
    a.ld = (uint32_t)(y_pitch ? y_pitch : n);
    a.K = (uint32_t)(k * eb);
    a.x_pitch = (uint32_t)(x_pitch * eb);
    a.w_pitch = (uint32_t)(w_pitch * eb);
    const bool words = y_fmt == kFmtWords;
    if (fmt == kFmtBF16) return words ? run_tiles<kFmtBF16, kFmtWords>(be, a) : run_tiles<kFmtBF16, kFmtBF16>(be, a);
    if (fmt == kFmtF16) return words ? run_tiles<kFmtF16, kFmtWords>(be, a) : run_tiles<kFmtF16, kFmtF16>(be, a);
    return words ? run_tiles<kFmtF8, kFmtWords>(be, a) : run_tiles<kFmtF8, kFmtF8>(be, a);
}

int launch_bf16_tiles(cg_backend *be, const void *x, uint32_t rows, const Weight &w, float *y) {
    if (!takes_bf16_tiles(rows, w)) return kDeclined;
    ProfScope prof(be, CG_K_GEMM_MFMA, 2.0 * (double)rows * w.n * w.k);
    return launch_narrow_tiles(be, kFmtBF16, x, w.k, rows, w.p, w.pitch, w.n, w.k, y, kFmtWords);
}

bool takes_bf16_tiles(uint32_t rows, const Weight &w) {
    return w.fmt == kFmtBF16 && reinterpret_cast<uintptr_t>(w.p) % 16 == 0 && fits_narrow_tiles(kFmtBF16, w.k, rows, w.pitch, w.n, w.k);
}

} // namespace cg
