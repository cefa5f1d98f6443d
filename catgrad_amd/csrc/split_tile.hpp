// 32-bit products on the bfloat16 matrix instructions, without loss of precision.
//
// A 32-bit float is the exact sum of three bfloat16 numbers (24 bits of significand = 3 x 8, each piece the nearest to what
// the ones before leave over), and products of bfloat16 numbers are exact in the matrix unit's 32-bit sums.  Of the nine
// piece products of x y the three of weight 2^-24 and below are left out; what the other six add up to is off by less than the
// rounding of one 32-bit multiplication (x y (1 + d), |d| <= 2^-23.4, and 2^-26 in the root mean square), and a chain over k
// rounds once per 16 values of k and piece instead of once per value.  Measured against 64 bits on 2048 values of k drawn from
// N(0, 1): relative error 7.0e-7 against 8.1e-7 of v_mfma_f32_32x32x2_f32 (8192: 1.5e-6 against 1.6e-6; all positive:
// 4.3e-7 against 6.5e-7).  Six instructions of 32 cycles for 16 values of k against eight of 64: 2.67 times the peak rate.
//
// The pieces share the 32-bit exponent's range but not infinity's company: a piece may round up to infinity beyond 3.38e38, and
// infinity times a zero piece is no number.  Values below 2^-126 lose bits of their lower pieces.  While it splits, a
// workgroup keeps the largest magnitude of every row of both operands, and a tile with a row at either end of the range (or
// an infinity) is multiplied again on the 32-bit instructions (plain_product).  So is a tile whose products could leave the range:
// the product of two first pieces may be above that of the values, and the products of the others, which are added first, have
// signs of their own and meet infinity alone.
#pragma once

#include "common.hpp"
#include "device_utils.hpp"

#include <type_traits>

namespace cg {
namespace split {

constexpr uint32_t kDepth = 16; // values of k per stage
typedef float float4v __attribute__((ext_vector_type(4)));
typedef float float2v __attribute__((ext_vector_type(2)));
typedef float float16v __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef uint32_t uint2v __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) char lds_char;

// [rows, K] operand of a tile.  k_fast: row r begins at p + row(r) and k is `s_k` apart; else rows are next to each other and
// k is s_k apart.
struct TileSide {
    const uint32_t *p;
    int64_t s_k;
};

// the six piece products, small ones first
constexpr int kPairA[6] = {0, 2, 1, 0, 1, 0}, kPairB[6] = {2, 0, 1, 1, 0, 0};

constexpr uint32_t lds_bytes(int bm, int bn) { return 2 * (uint32_t)(bm + bn) * kDepth * 6 + 64; }

__device__ __forceinline__ uint32_t cvt2(float x, float y) {
    const float2v v = {x, y};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}
__device__ __forceinline__ float lo2(uint32_t h) { return asf(h << 16); }
__device__ __forceinline__ float hi2(uint32_t h) { return asf(h & 0xFFFF0000u); }
// Two values' three pieces, two to a word.
__device__ __forceinline__ void split2(float x, float y, uint32_t (&w)[3]) {
    w[0] = cvt2(x, y);
    x -= lo2(w[0]), y -= hi2(w[0]);
    w[1] = cvt2(x, y);
    x -= lo2(w[1]), y -= hi2(w[1]);
    w[2] = cvt2(x, y);
}
__device__ __forceinline__ void grow(float &m, float x, float y) { // m = max(m, |x|, |y|)
    asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(m) : "v"(x), "v"(y));
}
// A row whose largest magnitude is m cannot be multiplied in pieces at full precision.
__device__ __forceinline__ bool out_of_range(float m) { return m > 3.0e38f || (m > 0.0f && m < 8.0e-28f); }
// Operands of magnitudes up to a and b: any number of products of their pieces adds up to less than 2^127.
__device__ __forceinline__ bool in_range(float a, float b) { return a * b < 0x1p95f; }
// the largest of a wave's values, none of them negative
template <int CTRL> __device__ __forceinline__ float with_lane(float m) {
    return fmaxf(m, asf((uint32_t)__builtin_amdgcn_update_dpp(0, (int)asu(m), CTRL, 0xF, 0xF, false)));
}
__device__ __forceinline__ float wave_max(float m) {
    m = with_lane<0x118>(with_lane<0x114>(with_lane<0x112>(with_lane<0x111>(m)))); // a row's 16 lanes: its last one has the largest
    m = with_lane<0x143>(with_lane<0x142>(m));                                       // the last lanes of rows to the rows behind
    return asf((uint32_t)__builtin_amdgcn_readlane((int)asu(m), 63));
}

// One operand's way into LDS: R rows, its share of a stage in registers, its pieces in fragment order.
//
// LDS: piece after piece, each R / 32 blocks of 32 rows x 16 k in the order in which the matrix instruction's lanes read them
// (lane group g = k / 8, 16 bytes a lane): 1 KB reads without bank conflicts.  The second lane group's rows sit elsewhere
// (row ^ 12), so that the 8-byte stores of four lanes that share a row meet no bank twice either (row ^ 8: 29 % of the LDS's cycles).
// k-contiguous: four lanes load a row's 16 values, 64 rows at a time.  Rows contiguous: a thread loads KQ x 4 values (KQ values
// of k, four rows) and turns them in registers.
template <int R, bool ROWS_FAST, int THREADS> struct Feed {
    static constexpr int STEP = THREADS / 4;                                // k contiguous: rows that a slot of all threads covers
    static constexpr int KQ = R / STEP;                                     // rows contiguous: values of k per thread
    static constexpr int SLOTS = R >= STEP ? R / STEP : 1;                  // 16-byte loads per thread and stage
    static constexpr int UNITS = ROWS_FAST ? 4 : SLOTS;                     // pieces of work between two stages
    static constexpr uint32_t PIECE = R * kDepth * 2;
    static_assert(!ROWS_FAST || KQ == 2 || KQ == 4, "a thread's share of a stage");
    uint32_t off[SLOTS]; // byte offsets of the 16-byte loads from the stage's first value
    uint32_t at;         // where this thread's pieces go
    float top[UNITS];    // largest magnitude per row seen
    float4v r[2][SLOTS];

    template <class Row> __device__ __forceinline__ void start(const TileSide &o, Row row, uint32_t last) {
        const uint32_t t = threadIdx.x;
#pragma unroll
        for (int u = 0; u < UNITS; u++) top[u] = 0.0f;
        if constexpr (!ROWS_FAST) {
            const uint32_t q = t % 4, l = t / 4;
#pragma unroll
            for (int h = 0; h < SLOTS; h++) off[h] = (uint32_t)(row(min(l + h * STEP, last)) * 4 + q * 16);
            at = (l / 32) * 1024 + (q / 2) * 512 + (((l % 32) ^ ((q / 2) * 12)) * 16) + (q % 2) * 8;
        } else {
            const uint32_t four = (t % 8) * 4, q = (t / 8) % (16 / KQ), block = t / (128 / KQ);
#pragma unroll
            for (int h = 0; h < SLOTS; h++) off[h] = (uint32_t)(row(min(block * 32 + four, last - last % 4)) * 4 + (uint64_t)(q * KQ + h) * o.s_k * 4);
            const uint32_t k = q * KQ, g = k / 8;
            at = block * 1024 + g * 512 + ((four ^ (g * 12)) * 16) + (k % 8) * 2;
        }
    }
    __device__ __forceinline__ void load(const TileSide &o, uint32_t stage, int set, int h) {
        const char *p = reinterpret_cast<const char *>(o.p) + (uint64_t)stage * (kDepth * 4) * (ROWS_FAST ? (uint64_t)o.s_k : 1ull);
        r[set][h] = *reinterpret_cast<const float4v *>(p + off[h]);
    }
    // the same where k may end within the stage or nothing is known of the alignment
    template <class Row> __device__ __forceinline__ void load_careful(const TileSide &o, Row row, uint32_t last, uint32_t K, uint32_t stage, int set, int h) {
        const uint32_t t = threadIdx.x;
        if constexpr (!ROWS_FAST) {
            const uint32_t k = stage * kDepth + (t % 4) * 4;
            const uint32_t *p = o.p + row(min(t / 4 + h * STEP, last));
#pragma unroll
            for (int i = 0; i < 4; i++) r[set][h][i] = asf(p[(int64_t)min(k + i, K - 1) * o.s_k]); // (no branches: the loads go out together)
#pragma unroll
            for (int i = 0; i < 4; i++) r[set][h][i] = k + i < K ? r[set][h][i] : 0.0f;
        } else {
            const uint32_t k = stage * kDepth + ((t / 8) % (16 / KQ)) * KQ + h, first = t / (128 / KQ) * 32 + (t % 8) * 4;
#pragma unroll
            for (int i = 0; i < 4; i++) r[set][h][i] = asf(o.p[(int64_t)min(k, K - 1) * o.s_k + row(min(first + i, last))]);
#pragma unroll
            for (int i = 0; i < 4; i++) r[set][h][i] = k < K ? r[set][h][i] : 0.0f;
        }
    }
    // splits unit u of a set into the stage at `lds`
    __device__ __forceinline__ void store(lds_char *lds, int set, int u) {
        if constexpr (!ROWS_FAST) {
            const float4v v = r[set][u];
            uint32_t a[3], b[3];
            split2(v[0], v[1], a);
            split2(v[2], v[3], b);
            grow(top[u], v[0], v[1]);
            grow(top[u], v[2], v[3]);
            if (R >= STEP || threadIdx.x < R * 4) {
#pragma unroll
                for (int p = 0; p < 3; p++) {
                    const uint2v w = {a[p], b[p]};
                    *reinterpret_cast<__attribute__((address_space(3))) uint2v *>(lds + p * PIECE + at + u * (STEP * 32)) = w;
                }
            }
        } else {
            uint32_t w[KQ / 2][3];
#pragma unroll
            for (int t = 0; t < KQ / 2; t++) {
                split2(r[set][2 * t][u], r[set][2 * t + 1][u], w[t]);
                grow(top[u], r[set][2 * t][u], r[set][2 * t + 1][u]);
            }
#pragma unroll
            for (int p = 0; p < 3; p++) {
                if constexpr (KQ == 4) {
                    const uint2v v = {w[0][p], w[1][p]};
                    *reinterpret_cast<__attribute__((address_space(3))) uint2v *>(lds + p * PIECE + at + u * 16) = v;
                } else {
                    *reinterpret_cast<__attribute__((address_space(3))) uint32_t *>(lds + p * PIECE + at + u * 16) = w[0][p];
                }
            }
        }
    }
    // any row out of the range that pieces cover (the lanes that share a row meet first)
    __device__ __forceinline__ bool bad() {
        bool b = false;
#pragma unroll
        for (int u = 0; u < UNITS; u++) {
            float m = top[u];
            if constexpr (!ROWS_FAST) {
                m = fmaxf(m, __shfl_xor(m, 1));
                m = fmaxf(m, __shfl_xor(m, 2));
            } else {
                m = fmaxf(m, __shfl_xor(m, 8));
                m = fmaxf(m, __shfl_xor(m, 16));
                if constexpr (KQ == 2) m = fmaxf(m, __shfl_xor(m, 32));
            }
            b |= out_of_range(m);
        }
        return b;
    }
    __device__ __forceinline__ float most() {
        float m = top[0];
#pragma unroll
        for (int u = 1; u < UNITS; u++) m = fmaxf(m, top[u]);
        return wave_max(m);
    }
};

// The 32-bit instructions on operands straight from memory: what is left for tiles that pieces do not cover.
template <int MT, int NT, bool AF, bool BF, class RowA, class RowB>
__device__ __forceinline__ void plain_product(float16v (&acc)[MT][NT], const TileSide &a, RowA row_a, uint32_t last_a, const TileSide &b, RowB row_b,
                                           uint32_t last_b, uint32_t K, uint32_t wm, uint32_t wn) {
    const uint32_t li = threadIdx.x % 32, lg = threadIdx.x % 64 / 32;
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[i][j][v] = 0.0f;
    for (uint32_t k = 0; k < K; k += 2) {
        const uint32_t kk = k + lg;
        float fa[MT], fb[NT];
#pragma unroll
        for (int i = 0; i < MT; i++) fa[i] = kk < K ? asf(a.p[(int64_t)kk * a.s_k + row_a(min(wm + i * 32 + li, last_a))]) : 0.0f;
#pragma unroll
        for (int j = 0; j < NT; j++) fb[j] = kk < K ? asf(b.p[(int64_t)kk * b.s_k + row_b(min(wn + j * 32 + li, last_b))]) : 0.0f;
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int j = 0; j < NT; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[i], fb[j], acc[i][j], 0, 0, 0);
    }
}

// acc = the workgroup's tile of A B^T: WM x WN waves of MT x NT blocks of 32 x 32 each (lane (li, lg), register v of a block: row
// 8 (v / 4) + 4 lg + v % 4, column li).  row_a / row_b: tile row -> element offset of that row; rows beyond last_a / last_b repeat
// the last one.
//
// A stage is 16 values of k.  While a stage is multiplied, the next one goes from registers through split2 into the other half of
// LDS and the one after it (two where a tile is small: LEAD) is asked for, a unit at a time between groups of NT matrix
// instructions; the fragments of a row of blocks are read while the row before it multiplies.  The barrier stands before the
// stage's last row: everybody has read the stage and written the next by then, whose fragments are read under that row.
template <int WM, int WN, int MT, int NT, bool AF, bool BF, bool CARE, class RowA, class RowB>
__device__ __forceinline__ void product(float16v (&acc)[MT][NT], lds_char *const lds, const TileSide &oa, RowA row_a, const uint32_t last_a, const TileSide &ob,
                                        RowB row_b, const uint32_t last_b, const uint32_t K) {
    constexpr int BM = 32 * WM * MT, BN = 32 * WN * NT;
    typedef Feed<BM, AF, 64 * WM * WN> FA;
    typedef Feed<BN, BF, 64 * WM * WN> FB;
    constexpr int LEAD = FA::SLOTS + FB::SLOTS > 4 ? 1 : 2;
    constexpr uint32_t STAGE = 3 * (FA::PIECE + FB::PIECE);
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64, li = lane % 32, lg = lane / 32;
    const uint32_t bma = wave / WN * MT, bnb = wave % WN * NT; // this wave's first block of rows and of columns
    const uint32_t fl = lg * 512 + ((li ^ (lg * 12)) * 16);
    lds_char *const fa_base = lds + bma * 1024 + fl, *const fb_base = lds + 3 * FA::PIECE + bnb * 1024 + fl;
    FA fa;
    FB fb;
    fa.start(oa, row_a, last_a);
    fb.start(ob, row_b, last_b);
    const uint32_t nk = CARE ? (K + kDepth - 1) / kDepth : K / kDepth; // stages of the loop (CARE: with the last, ragged one)
    // (behind the last stage the last one is asked for again: one way through the loop, and values that nobody multiplies)
    auto ask_a = [&](uint32_t s, int set, int h) {
        if constexpr (CARE) fa.load_careful(oa, row_a, last_a, K, s, set, h);
        else fa.load(oa, min(s, nk - 1), set, h);
    };
    auto ask_b = [&](uint32_t s, int set, int h) {
        if constexpr (CARE) fb.load_careful(ob, row_b, last_b, K, s, set, h);
        else fb.load(ob, min(s, nk - 1), set, h);
    };
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[i][j][v] = 0.0f;
    auto meet = [&]() {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0xC07F); // lgkmcnt(0)
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    constexpr int AS = MT > 1 ? 2 : 1;
    bf16x8 a[AS][3], b[NT][3];
    auto read = [&](lds_char *p) { return __builtin_bit_cast(bf16x8, *reinterpret_cast<__attribute__((address_space(3))) float4v *>(p)); };
    auto read_a = [&](const int par, const int i, const int p) { a[i % AS][p] = read(fa_base + par * STAGE + p * FA::PIECE + i * 1024); };
    auto read_b = [&](const int par, const int j, const int p) { b[j][p] = read(fb_base + par * STAGE + p * FB::PIECE + j * 1024); };
    // One stage (PAR: its half of LDS): the small products first.
    auto stage = [&](const uint32_t s, auto par_) {
        constexpr int PAR = decltype(par_)::value;
        constexpr int SET = LEAD == 2 ? (PAR + 1) % 2 : 0; // registers of stage s + 1, to be filled with stage s + 1 + LEAD
        constexpr int UNITS = FA::UNITS + FB::UNITS, GROUPS = MT > 1 ? (MT - 1) * 6 : 6;
        lds_char *const to = lds + (PAR ^ 1) * STAGE;
        auto unit = [&](const int u) {
            if (u < FA::UNITS) {
                fa.store(to, SET, u);
                if (!AF) ask_a(s + 1 + LEAD, SET, u);
                else if (u == 3)
                    for (int h = 0; h < FA::SLOTS; h++) ask_a(s + 1 + LEAD, SET, h);
            } else {
                const int v = u - FA::UNITS;
                fb.store(to + 3 * FA::PIECE, SET, v);
                if (!BF) ask_b(s + 1 + LEAD, SET, v);
                else if (v == 3)
                    for (int h = 0; h < FB::SLOTS; h++) ask_b(s + 1 + LEAD, SET, h);
            }
        };
#pragma unroll
        for (int i = 0; i < MT; i++) {
            if (MT > 1 && i == MT - 1) meet();
#pragma unroll
            for (int g = 0; g < 6; g++) {
#pragma unroll
                for (int j = 0; j < NT; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i % AS][kPairA[g]], b[j][kPairB[g]], acc[i][j], 0, 0, 0);
                const int group = i * 6 + g;
                if (group < GROUPS) {
#pragma unroll
                    for (int u = 0; u < UNITS; u++)
                        if (u * GROUPS / UNITS == group) unit(u);
                }
                if (MT > 1) {
                    if (g < 3) {
                        if (i + 1 < MT) read_a(PAR, i + 1, kPairA[g]);
                        else read_a(PAR ^ 1, 0, kPairA[g]);
                    }
                    if (i == MT - 1) {
                        const int gone = g == 0 ? 2 : g == 3 ? 1 : g == 5 ? 0 : -1; // the piece of B that was used for the last time
                        if (gone >= 0) {
#pragma unroll
                            for (int j = 0; j < NT; j++) read_b(PAR ^ 1, j, gone);
                        }
                    }
                }
                if constexpr (!CARE) {
#pragma unroll
                    for (int j = 0; j < NT; j++) { // what goes along, between the matrix instructions
                        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
                        __builtin_amdgcn_sched_group_barrier(0x002, 24 / NT + 1, 0);
                        __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if (MT == 1) {
            meet();
#pragma unroll
            for (int p = 0; p < 3; p++) read_a(PAR ^ 1, 0, p);
#pragma unroll
            for (int p = 0; p < 3; p++)
#pragma unroll
                for (int j = 0; j < NT; j++) read_b(PAR ^ 1, j, p);
        }
    };
    typedef std::integral_constant<int, 0> P0;
    typedef std::integral_constant<int, 1> P1;
    if (nk) {
        for (int h = 0; h < FA::SLOTS; h++) ask_a(0, 0, h);
        for (int h = 0; h < FB::SLOTS; h++) ask_b(0, 0, h);
        if constexpr (LEAD == 2) {
            for (int h = 0; h < FA::SLOTS; h++) ask_a(1, 1, h);
            for (int h = 0; h < FB::SLOTS; h++) ask_b(1, 1, h);
        }
#pragma unroll
        for (int u = 0; u < FA::UNITS; u++) fa.store(lds, 0, u);
#pragma unroll
        for (int u = 0; u < FB::UNITS; u++) fb.store(lds + 3 * FA::PIECE, 0, u);
        for (int h = 0; h < FA::SLOTS; h++) ask_a(LEAD, 0, h);
        for (int h = 0; h < FB::SLOTS; h++) ask_b(LEAD, 0, h);

        meet();
#pragma unroll
        for (int p = 0; p < 3; p++) read_a(0, 0, p);
#pragma unroll
        for (int p = 0; p < 3; p++)
#pragma unroll
            for (int j = 0; j < NT; j++) read_b(0, j, p);
        for (uint32_t s = 0;; s += 2) {
            stage(s, P0{});
            if (s + 1 >= nk) break;
            stage(s + 1, P1{});
            if (s + 2 >= nk) break;
        }
    }
    if (MT * NT < 8 && !CARE && K % kDepth) { // what is left of k, a stage by itself (the wide tile has no registers for it)
#pragma unroll
        for (int h = 0; h < FA::SLOTS; h++) fa.load_careful(oa, row_a, last_a, K, nk, 0, h);
#pragma unroll
        for (int h = 0; h < FB::SLOTS; h++) fb.load_careful(ob, row_b, last_b, K, nk, 0, h);
        meet(); // (nobody reads the half that is written now)
#pragma unroll
        for (int u = 0; u < FA::UNITS; u++) fa.store(lds, 0, u);
#pragma unroll
        for (int u = 0; u < FB::UNITS; u++) fb.store(lds + 3 * FA::PIECE, 0, u);
        meet();
#pragma unroll
        for (int p = 0; p < 3; p++)
#pragma unroll
            for (int j = 0; j < NT; j++) read_b(0, j, p);
#pragma unroll
        for (int i = 0; i < MT; i++) {
#pragma unroll
            for (int p = 0; p < 3; p++) read_a(0, i, p);
#pragma unroll
            for (int g = 0; g < 6; g++)
#pragma unroll
                for (int j = 0; j < NT; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i % AS][kPairA[g]], b[j][kPairB[g]], acc[i][j], 0, 0, 0);
        }
    }

    __attribute__((address_space(3))) float2v *const tops = reinterpret_cast<__attribute__((address_space(3))) float2v *>(lds + 2 * STAGE);
    const bool bad_a = fa.bad(), bad_b = fb.bad(); // (both: every lane takes part in the exchanges)
    const bool some = __builtin_amdgcn_ballot_w64(bad_a || bad_b) != 0;
    const float2v top = {some ? INFINITY : fa.most(), fb.most()};
    if (lane == 0) tops[wave] = top;
    meet();
    float2v most = tops[0];
#pragma unroll
    for (int w = 1; w < WM * WN; w++) most = {fmaxf(most[0], tops[w][0]), fmaxf(most[1], tops[w][1])};
    if (most[0] == INFINITY || !in_range(most[0], most[1])) plain_product<MT, NT, AF, BF>(acc, oa, row_a, last_a, ob, row_b, last_b, K, bma * 32, bnb * 32);
}

} // namespace split
} // namespace cg
