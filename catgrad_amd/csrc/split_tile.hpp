// 32-bit products on the bfloat16 matrix instructions, without loss of precision.
//
// A 32-bit float is the exact sum of three bfloat16 numbers (24 bits of significand = 3 x 8, each piece the nearest to what
// the ones before leave over), and products of bfloat16 numbers are exact in the matrix unit's 32-bit sums.  Of the nine
// piece products of x y the three of weight 2^-25 and below are left out: together at most 2^-24.0 of |x y|, which is the
// largest rounding of one 32-bit multiplication, and 2^-27.5 in the root mean square, a fifth of that rounding's.
//
// The matrix instruction cuts what it adds off towards minus infinity below its sum's last bits, so a chain of them over all of k
// moves every output, of either sign, to the same side (by 8e-8 of their root mean square at 2048 values of k), which does not
// average out over a model's rows and layers as roundings do.  The six piece products of 16 values of k are therefore a chain of
// their own that starts from zero, of the negated left operand for every other 16, and a vector instruction adds its sum to the
// total or takes it away: one rounding to nearest per 16 values of k, where the 32-bit matrix instructions round 8 times.
// Both operands are multiplied by 2^16 on their way into pieces, and the chains' sums by 2^-32 as they are added: then the three
// pieces of every 32-bit number, the subnormal ones included, are bfloat16 numbers (multiples of 2^-133).  What the pieces do
// not hold are infinities and products at the upper end of the range: while it splits, a workgroup keeps the largest magnitude of
// either operand, and a tile whose products could leave the range is multiplied again on the 32-bit instructions (`plain`).
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

// the six piece products, the largest last, in an order that is done with the left side's small pieces early
constexpr int kPairA[6] = {2, 1, 1, 0, 0, 0}, kPairB[6] = {0, 1, 0, 2, 1, 0};

constexpr uint32_t kPitch = kDepth + 4; // words from row to row where a stage lies in LDS in 32 bits
constexpr uint32_t lds_bytes(int bm, int bn) { return 2 * (uint32_t)(bm + bn) * kDepth * 6 + 64; }

__device__ __forceinline__ uint32_t cvt2(float x, float y) {
    const float2v v = {x, y};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}
constexpr float kUp = 65536.0f, kDown = 1.0f / (65536.0f * 65536.0f); // both operands' scale, and the products' way back
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
// Operands of magnitudes up to a and b: 16 products of scaled pieces stay below 2^127.
__device__ __forceinline__ bool in_range(float a, float b) { return a < 0x1p110f && b < 0x1p110f && a * b < 0x1p90f; }
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
    float top;           // largest magnitude seen
    float4v r[2][SLOTS];

    template <class Row> __device__ __forceinline__ void start(const TileSide &o, Row row, uint32_t last) {
        const uint32_t t = threadIdx.x;
        top = 0.0f;
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
    // splits unit u of a set, times `up`, into the stage at `lds`
    __device__ __forceinline__ void store(lds_char *lds, int set, int u, float up) {
        if constexpr (!ROWS_FAST) {
            const float4v v = r[set][u];
            uint32_t a[3], b[3];
            split2(v[0] * up, v[1] * up, a);
            split2(v[2] * up, v[3] * up, b);
            grow(top, v[0], v[1]);
            grow(top, v[2], v[3]);
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
                split2(r[set][2 * t][u] * up, r[set][2 * t + 1][u] * up, w[t]);
                grow(top, r[set][2 * t][u], r[set][2 * t + 1][u]);
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
    // the values of a set as they are, rows of kPitch
    __device__ __forceinline__ void store_plain(__attribute__((address_space(3))) float *lds, int set) {
        const uint32_t t = threadIdx.x;
        if constexpr (!ROWS_FAST) {
#pragma unroll
            for (int h = 0; h < SLOTS; h++)
                if (R >= STEP || t < R * 4) *reinterpret_cast<__attribute__((address_space(3))) float4v *>(lds + (t / 4 + h * STEP) * kPitch + t % 4 * 4) = r[set][h];
        } else {
            const uint32_t row = t / (128 / KQ) * 32 + t % 8 * 4, k = t / 8 % (16 / KQ) * KQ;
#pragma unroll
            for (int h = 0; h < SLOTS; h++)
#pragma unroll
                for (int i = 0; i < 4; i++) lds[(row + i) * kPitch + k + h] = r[set][h][i];
        }
    }
};

// acc = the workgroup's tile of A B^T: WM x WN waves of MT x NT blocks of 32 x 32 each (lane (li, lg), register v of a block: row
// 8 (v / 4) + 4 lg + v % 4, column li).  row_a / row_b: tile row -> element offset of that row; rows beyond last_a / last_b repeat
// the last one.
//
// A stage is 16 values of k.  While a stage is multiplied, the next one goes from registers through split2 into the other half of
// LDS and the one after it (two where a tile is small: LEAD) is asked for, a unit at a time between the matrix instructions; the
// fragments of a row of blocks are read while the row before it multiplies.  A block's chain of six is added to its total while the
// next block's chain runs (SETS: the registers for that; the wide tile has none and waits, which its other wave on the SIMD
// fills).  The barrier stands before the stage's last row: everybody has read the stage and written the next by then, whose
// fragments are read under that row.
// Up to four values of k are multiplied by the 32-bit instructions alone, which lose less of so short a sum.
template <int WM, int WN, int MT, int NT, bool AF, bool BF, bool CARE, class RowA, class RowB>
__device__ __forceinline__ void product(float16v (&acc)[MT][NT], lds_char *const lds, const TileSide &oa, RowA row_a, const uint32_t last_a, const TileSide &ob,
                                        RowB row_b, const uint32_t last_b, const uint32_t K) {
    constexpr int BM = 32 * WM * MT, BN = 32 * WN * NT;
    typedef Feed<BM, AF, 64 * WM * WN> FA;
    typedef Feed<BN, BF, 64 * WM * WN> FB;
    constexpr int LEAD = FA::SLOTS + FB::SLOTS > 4 ? 1 : 2;
    constexpr bool WIDE = MT * NT >= 8;
    constexpr int TOGETHER = WIDE ? 1 : NT;                            // blocks of a row whose chains run side by side
    constexpr int GROUPS = MT * NT / TOGETHER, SETS = WIDE ? 1 : 2;    // of such chains in a stage; of their sums in registers
    constexpr bool CARRY = GROUPS == 1;                                // a stage's sums are added in the next stage
    constexpr uint32_t STAGE = 3 * (FA::PIECE + FB::PIECE);
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64, li = lane % 32, lg = lane / 32;
    const uint32_t bma = wave / WN * MT, bnb = wave % WN * NT; // this wave's first block of rows and of columns
    const uint32_t fl = lg * 512 + ((li ^ (lg * 12)) * 16);
    lds_char *const fa_base = lds + bma * 1024 + fl, *const fb_base = lds + 3 * FA::PIECE + bnb * 1024 + fl;
    FA fa;
    FB fb;
    fa.start(oa, row_a, last_a);
    fb.start(ob, row_b, last_b);
    const uint32_t nk = K <= 4 ? 0 : CARE ? (K + kDepth - 1) / kDepth : K / kDepth; // stages of the loop (CARE: with the last, ragged one)
    // (behind the last stage the last one is asked for again: one way through the loop, and values that nobody multiplies)
    auto ask_a = [&](uint32_t s, int set, int h) {
        if constexpr (CARE) fa.load_careful(oa, row_a, last_a, K, s, set, h);
        else fa.load(oa, min(s, nk - 1), set, h);
    };
    auto ask_b = [&](uint32_t s, int set, int h) {
        if constexpr (CARE) fb.load_careful(ob, row_b, last_b, K, s, set, h);
        else fb.load(ob, min(s, nk - 1), set, h);
    };
    const float16v zero = {};
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < NT; j++) acc[i][j] = zero;
    auto meet = [&]() {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0xC07F); // lgkmcnt(0)
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    constexpr int AS = MT > 1 && !WIDE ? 2 : 1; // (the wide tile reads the left side's next fragments under a row's last chain)
    bf16x8 a[AS][3], b[NT][3];
    auto read = [&](lds_char *p) { return __builtin_bit_cast(bf16x8, *reinterpret_cast<__attribute__((address_space(3))) float4v *>(p)); };
    auto read_a = [&](const int par, const int i, const int p) { a[i % AS][p] = read(fa_base + par * STAGE + p * FA::PIECE + i * 1024); };
    auto read_b = [&](const int par, const int j, const int p) { b[j][p] = read(fb_base + par * STAGE + p * FB::PIECE + j * 1024); };
    float16v sum[SETS][TOGETHER]; // chains of six
    if (CARRY)
        for (int t = 0; t < TOGETHER; t++) sum[SETS - 1][t] = zero;
    auto add = [&](const int group, const int set, const float down) {
#pragma unroll
        for (int t = 0; t < TOGETHER; t++) {
            float16v &to = acc[group * TOGETHER / NT][group * TOGETHER % NT + t];
#pragma unroll
            for (int v = 0; v < 16; v++) to[v] = __builtin_fmaf(sum[set][t][v], down, to[v]);
        }
    };
    // One stage (PAR: its half of LDS, 1: its left operand is negated)
    auto stage = [&](const uint32_t s, auto par_) {
        constexpr int PAR = decltype(par_)::value;
        constexpr int SET = LEAD == 2 ? (PAR + 1) % 2 : 0; // registers of stage s + 1, to be filled with stage s + 1 + LEAD
        constexpr int UNITS = FA::UNITS + FB::UNITS, SLOTS = (MT > 1 ? MT - 1 : 1) * NT / TOGETHER * 6; // places between the matrix instructions before the barrier
        constexpr float down = PAR ? -kDown : kDown;
        lds_char *const to = lds + (PAR ^ 1) * STAGE;
        auto unit = [&](const int u) {
            if (u < FA::UNITS) {
                fa.store(to, SET, u, PAR ? kUp : -kUp);
                if (!AF) ask_a(s + 1 + LEAD, SET, u);
                else if (u == 3)
                    for (int h = 0; h < FA::SLOTS; h++) ask_a(s + 1 + LEAD, SET, h);
            } else {
                const int v = u - FA::UNITS;
                fb.store(to + 3 * FA::PIECE, SET, v, kUp);
                if (!BF) ask_b(s + 1 + LEAD, SET, v);
                else if (v == 3)
                    for (int h = 0; h < FB::SLOTS; h++) ask_b(s + 1 + LEAD, SET, h);
            }
        };
#pragma unroll
        for (int group = 0; group < GROUPS; group++) {
            const int i = group * TOGETHER / NT, j0 = group * TOGETHER % NT, set = (PAR * GROUPS + group) % SETS, before = (set + 1) % SETS;
            if (MT > 1 && i == MT - 1 && j0 == 0) meet();
#pragma unroll
            for (int g = 0; g < 6; g++) {
#pragma unroll
                for (int t = 0; t < TOGETHER; t++)
                    sum[set][t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i % AS][kPairA[g]], b[j0 + t][kPairB[g]], g ? sum[set][t] : zero, 0, 0, 0);
                if (SETS == 2 && g == 4 && (group || CARRY)) add(group ? group - 1 : GROUPS - 1, before, group ? down : -down);
                const int slot = group * 6 + g;
                if (slot < SLOTS) {
#pragma unroll
                    for (int u = 0; u < UNITS; u++)
                        if (u * SLOTS / UNITS == slot) unit(u);
                }
                if (MT > 1) {
                    const int next = (i + 1) % MT, par = i + 1 < MT ? PAR : PAR ^ 1;
                    if (WIDE ? j0 + TOGETHER == NT && (g == 0 || g == 2 || g == 5) : j0 == 0 && g < 3) read_a(par, next, WIDE ? kPairA[g] : g);
                    if (i == MT - 1 && g >= 3) { // (used for the last time)
#pragma unroll
                        for (int t = 0; t < TOGETHER; t++) read_b(PAR ^ 1, j0 + t, kPairB[g]);
                    }
                }
                if (MT * NT < 4) __builtin_amdgcn_sched_barrier(0); // (or all of a unit's work would stand behind the chain)
            }
            if (WIDE) add(group, 0, down);
            if constexpr (!CARE && MT * NT >= 4) {
#pragma unroll
                for (int g = 0; g < 6 * TOGETHER; g++) { // what goes along, between the matrix instructions
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, WIDE ? 6 : 8, 0);
                    __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if (SETS == 2 && !CARRY) add(GROUPS - 1, (PAR * GROUPS + GROUPS - 1) % SETS, down);
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
        for (int u = 0; u < FA::UNITS; u++) fa.store(lds, 0, u, kUp);
#pragma unroll
        for (int u = 0; u < FB::UNITS; u++) fb.store(lds + 3 * FA::PIECE, 0, u, kUp);
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
            if (s + 1 >= nk) {
                if (CARRY) add(0, 0, kDown);
                break;
            }
            stage(s + 1, P1{});
            if (s + 2 >= nk) {
                if (CARRY) add(0, SETS - 1, -kDown);
                break;
            }
        }
    }
    if (MT * NT < 8 && !CARE && K > 4 && K % kDepth) { // what is left of k, a stage by itself (the wide tile has no registers for it)
#pragma unroll
        for (int h = 0; h < FA::SLOTS; h++) fa.load_careful(oa, row_a, last_a, K, nk, 0, h);
#pragma unroll
        for (int h = 0; h < FB::SLOTS; h++) fb.load_careful(ob, row_b, last_b, K, nk, 0, h);
        meet(); // (nobody reads the half that is written now)
#pragma unroll
        for (int u = 0; u < FA::UNITS; u++) fa.store(lds, 0, u, nk % 2 ? -kUp : kUp);
#pragma unroll
        for (int u = 0; u < FB::UNITS; u++) fb.store(lds + 3 * FA::PIECE, 0, u, kUp);
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
            for (int j = 0; j < NT; j++) {
                float16v &t = sum[0][j % TOGETHER];
#pragma unroll
                for (int g = 0; g < 6; g++) t = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i % AS][kPairA[g]], b[j][kPairB[g]], g ? t : zero, 0, 0, 0);
#pragma unroll
                for (int v = 0; v < 16; v++) acc[i][j][v] = __builtin_fmaf(t[v], nk % 2 ? -kDown : kDown, acc[i][j][v]);
            }
        }
    }

    uint32_t plain = K <= 4;
    if (!plain) {
        __attribute__((address_space(3))) float2v *const tops = reinterpret_cast<__attribute__((address_space(3))) float2v *>(lds + 2 * STAGE);
        const float2v top = {wave_max(fa.top), wave_max(fb.top)};
        if (lane == 0) tops[wave] = top;
        meet();
        float2v most = tops[0];
#pragma unroll
        for (int w = 1; w < WM * WN; w++) most = {fmaxf(most[0], tops[w][0]), fmaxf(most[1], tops[w][1])};
        plain = !in_range(most[0], most[1]);
    }
    if (!__builtin_amdgcn_readfirstlane(plain)) return;
    // The 32-bit instructions, for what the pieces do not hold: a stage is multiplied while the next one is on its way.  Lane group
    // lg multiplies k = 8 c + 4 lg + t in the t-th of four instructions.
    typedef __attribute__((address_space(3))) float lds_float;
    lds_float *const whole = (lds_float *)lds;
    constexpr uint32_t WHOLE = (BM + BN) * kPitch;
    static_assert(2 * WHOLE * 4 <= 2 * STAGE, "both stages fit where the pieces were");
    const uint32_t stages = (K + kDepth - 1) / kDepth;
    auto fetch = [&](const uint32_t s) {
        if (CARE || (s + 1) * kDepth > K) {
#pragma unroll
            for (int h = 0; h < FA::SLOTS; h++) fa.load_careful(oa, row_a, last_a, K, s, 0, h);
#pragma unroll
            for (int h = 0; h < FB::SLOTS; h++) fb.load_careful(ob, row_b, last_b, K, s, 0, h);
        } else {
#pragma unroll
            for (int h = 0; h < FA::SLOTS; h++) fa.load(oa, s, 0, h);
#pragma unroll
            for (int h = 0; h < FB::SLOTS; h++) fb.load(ob, s, 0, h);
        }
    };
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < NT; j++) acc[i][j] = zero;
    fetch(0);
    meet(); // (everybody is done with the pieces)
    for (uint32_t s = 0; s < stages; s++) {
        lds_float *const at = whole + s % 2 * WHOLE;
        fa.store_plain(at, 0);
        fb.store_plain(at + BM * kPitch, 0);
        meet(); // (the stage is there, and nobody reads the one before the last)
        fetch(min(s + 1, stages - 1));
#pragma unroll
        for (int c = 0; c < 2; c++) {
            float4v x[MT], y[NT];
#pragma unroll
            for (int i = 0; i < MT; i++) x[i] = *reinterpret_cast<__attribute__((address_space(3))) float4v *>(at + ((bma + i) * 32 + li) * kPitch + c * 8 + lg * 4);
#pragma unroll
            for (int j = 0; j < NT; j++) y[j] = *reinterpret_cast<__attribute__((address_space(3))) float4v *>(at + (BM + (bnb + j) * 32 + li) * kPitch + c * 8 + lg * 4);
#pragma unroll
            for (int t = 0; t < 4; t++)
#pragma unroll
                for (int i = 0; i < MT; i++)
#pragma unroll
                    for (int j = 0; j < NT; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(x[i][t], y[j][t], acc[i][j], 0, 0, 0);
        }
    }
}

} // namespace split
} // namespace cg
