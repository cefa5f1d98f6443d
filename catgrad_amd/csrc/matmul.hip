// Batched matrix multiply for gfx950: C[b, M, N] = A[b, M, K] * B[b, K, N], f32.
//
// Operands are consumed through their strides: row/column strides of A and B are
// arbitrary (transposed views cost nothing), every batch axis has its own stride per
// operand (0 = shared), so `linear`'s transposed, batch-broadcast weight view
// (catgrad/src/stdlib/nn/mod.rs:182-204) and attention's [B, h, S, hd] head views
// (catgrad-llm-models/src/models/llama.rs:285-345) are multiplied in place.  When the
// right-hand side is shared by the whole batch and the left-hand side's batch and row
// axes form one run, the batch is folded into M (one tall GEMM instead of B small ones).
//
// Kernels
//   split_gemm_kernel  (split_gemm.hip) every f32 product of more than eight rows.
//   narrow_tile_kernel (block_products.hip) products of the narrow dtypes with an operand that lies in memory as
//                      patterns, on 128-wide tiles (narrow_route.hpp decides).
//   mfma_gemm_kernel   the other products of the narrow dtypes: 256 threads = 2x2 waves, 128x128x32 macro tiles (2x2
//                      32x32 accumulators per wave) or, with enough of them (one per two compute units for the 16-bit
//                      dtypes, one per unit for fp8), 256x256x32 (each wave a 128x128 block as 4x4 accumulators, all 256
//                      accumulation registers, 144 KiB of LDS), fed by loads straight into LDS where k is whole turns
//                      of the ring (mfma_gemm_dlds_kernel).  Tiles of words are narrowed to bf16 / f16 on their way into LDS (fp8 words to
//                      bf16, which holds them exactly), or operands lie narrow in memory (pack_operand_kernel);
//                      v_mfma_f32_32x32x16_{bf16,f16} / v_mfma_scale_f32_32x32x64_f8f6f4.  Staged K-fastest in
//                      LDS; whole tiles are loaded at fixed per-lane offsets without tests; two LDS buffers,
//                      next tile's global loads in flight during the MFMAs, XCD-aware tile order.
//                      MFMA-bound: 2*M*N*K flop.
//   skinny_kt_*        M <= 8 with K-contiguous B rows (decode-time linear layers and q.K^T),
//                      HBM-bound streams of B (4*K*N bytes):
//                      skinny_kt_wide / _narrow: a wave per output column (or per 4 columns, or a
//                      column per 16/32 lanes for short K), 16-byte loads along K, wave shuffle
//                      reduction;
//                      skinny_kt_mfma_xreg: batches of them, and products alone that skinny_alone leaves here, on the
//                      4x4x1 matrix instruction with the activations held in registers; others: skinny.hpp.
//   skinny_nn_kernel   M <= 8 with N-contiguous B rows (p.V of a decode step), split over K
//                      with a second pass that adds the partial sums.
//   simple_gemm_kernel u32 (wrapping) and any shape the others decline.
//
// Accumulation is f32 with fused multiply-add; the summation order differs from the
// reference's `matrixmultiply::sgemm`, which is why the contract for matmul is 1e-3
// relative (ndarray.rs:750-816 makes no promise on order either).
#include "gemm_args.hpp"
#include "skinny.hpp"

#include <algorithm>
#include <type_traits>

namespace cg {

namespace {

// ------------------------------------------------------------------------------------------
// MFMA kernel
// ------------------------------------------------------------------------------------------
constexpr int BM = 128, BK = 32; // (the kernels shadow BM and define BN from their tile parameters)
constexpr int PITCH = BK + 4; // words per LDS row: row r starts at bank 4r mod 32
constexpr size_t gemm_lds_bytes(int bn, int bm = BM, bool half = false) {
    return 2 * (size_t)(bm + bn) * (half ? BK / 2 + 4 : PITCH) * sizeof(float);
}
constexpr int kThreads = 256;
constexpr uint32_t kXcds = 8, kGroupM = 8;

typedef float float4v __attribute__((ext_vector_type(4)));
typedef float float16v __attribute__((ext_vector_type(16)));

// Loads one TR x BK tile (rows along `R` with stride s_r, k with stride s_k) into
// registers: TR*BK/4/256 float4 slots per thread.  Layout of the float4 slots of a tile:
//   K-contiguous source (s_k == 1): slot = row*(BK/4) + kq  (float4 along k; 8 lanes read
//                                                            128 contiguous bytes of a row)
//   R-contiguous source (s_r == 1): float4 along rows; a wave's 64 slots are 16 row-quads x 4 values of k
//                                   (rows_fast_slot), so that its LDS stores spread over all banks
//   otherwise                      : as K-contiguous, element by element
template <int TR> struct TileRegs {
    static constexpr int slots = TR * BK / 4 / 256;
    float4v v[slots];
};

__device__ __forceinline__ float ld_guard(const uint32_t *p, bool ok) { return ok ? asf(*p) : 0.0f; }

// Slot -> (first of four rows, k) of a tile whose rows are the unit-stride axis in memory: 16 row-quads x 4 consecutive k
// per wave, global loads of 256 contiguous bytes per k.  An f32 tile keeps that order in LDS (store_tile).  A tile that is
// narrowed to 16 bits is staged K-fastest (pairs of k share a word), so a lane's four values go to four different LDS
// rows, one store each; with each lane writing its four rows in an order rotated by its row-quad (rows_fast_order), a
// wave's store covers all 32 banks twice, which is the best 64 lanes can do (a whole wave on one k would hit 2 banks).
template <int TR> __device__ __forceinline__ void rows_fast_slot(uint32_t slot, uint32_t &row, uint32_t &k) {
    const uint32_t group = slot / 64, in = slot % 64;
    row = (group % (TR / 64)) * 64 + (in % 16) * 4;
    k = (group / (TR / 64)) * 4 + in / 16;
}
__device__ __forceinline__ uint32_t rows_fast_order(uint32_t slot, int i) { return ((uint32_t)i + ((slot % 16) >> 1)) & 3u; }
__device__ __forceinline__ float pick4(const float4v &v, uint32_t j) { return j == 0 ? v[0] : j == 1 ? v[1] : j == 2 ? v[2] : v[3]; }

template <bool ROWS_FAST, int TR>
__device__ __forceinline__ void load_tile(TileRegs<TR> &t, const uint32_t *base, int64_t s_r, int64_t s_k, uint32_t r0,
                                          uint32_t k0, uint32_t R, uint32_t K, bool vec_ok) {
#pragma unroll
    for (int h = 0; h < TileRegs<TR>::slots; h++) {
        uint32_t slot = threadIdx.x + h * kThreads;
        if (!ROWS_FAST) {
            uint32_t row = r0 + slot / (BK / 4), k = k0 + (slot % (BK / 4)) * 4;
            const uint32_t *p = base + (int64_t)row * s_r + (int64_t)k * s_k;
            if (vec_ok && row < R && k + 3 < K) {
                t.v[h] = *reinterpret_cast<const float4v *>(p);
            } else {
                bool rok = row < R;
                t.v[h][0] = ld_guard(p, rok && k < K);
                t.v[h][1] = ld_guard(p + s_k, rok && k + 1 < K);
                t.v[h][2] = ld_guard(p + 2 * s_k, rok && k + 2 < K);
                t.v[h][3] = ld_guard(p + 3 * s_k, rok && k + 3 < K);
            }
        } else {
            uint32_t row, k;
            rows_fast_slot<TR>(slot, row, k);
            row += r0;
            k += k0;
            const uint32_t *p = base + (int64_t)row * s_r + (int64_t)k * s_k;
            if (vec_ok && k < K && row + 3 < R) {
                t.v[h] = *reinterpret_cast<const float4v *>(p);
            } else {
                bool kok = k < K;
                t.v[h][0] = ld_guard(p, kok && row < R);
                t.v[h][1] = ld_guard(p + s_r, kok && row + 1 < R);
                t.v[h][2] = ld_guard(p + 2 * s_r, kok && row + 2 < R);
                t.v[h][3] = ld_guard(p + 3 * s_r, kok && row + 3 < R);
            }
        }
    }
}

// Stores the registers of a k-contiguous operand into an LDS tile, [TR][PITCH].
template <int TR> __device__ __forceinline__ void store_tile(const TileRegs<TR> &t, float *lds) {
#pragma unroll
    for (int h = 0; h < TileRegs<TR>::slots; h++) {
        uint32_t slot = threadIdx.x + h * kThreads;
        uint32_t row = slot / (BK / 4), k = (slot % (BK / 4)) * 4;
        *reinterpret_cast<float4v *>(lds + row * PITCH + k) = t.v[h];
    }
}

// ---- the 16-bit float dtypes on their own matrix instructions ------------------------------------------------
// Tensors of these dtypes hold f32 words with exactly representable values, so a tile is narrowed to its 16-bit
// patterns on the way into LDS (exact: the upper half of the word for bfloat16, v_cvt_f16_f32 for binary16) and the
// products run on v_mfma_f32_32x32x16_{bf16,f16}: 16 k per instruction instead of 2, f32 accumulation as before.
// LDS rows hold BK/2 words + 4 of padding (a row starts 20 banks after the one before: 8 lanes of a 128-bit
// read cover all 32 banks); a lane's 128-bit read is its 8 consecutive k of one 16-deep chunk.
constexpr int PITCH_H = BK / 2 + 4;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef long long2v __attribute__((ext_vector_type(2)));
typedef float float2v __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef uint32_t uint4v __attribute__((ext_vector_type(4)));
typedef int int4v __attribute__((ext_vector_type(4)));
typedef int int8v __attribute__((ext_vector_type(8)));

// HALF: 1 bfloat16, 2 binary16
template <int HALF> __device__ __forceinline__ uint32_t pack_halves(float lo, float hi) {
    if constexpr (HALF == 1) return (asu(lo) >> 16) | (asu(hi) & 0xFFFF0000u);
    return (uint32_t)__half_as_ushort(__float2half_rn(lo)) | ((uint32_t)__half_as_ushort(__float2half_rn(hi)) << 16);
}
template <int HALF> __device__ __forceinline__ uint16_t narrow_half(float v) {
    if constexpr (HALF == 1) return (uint16_t)(asu(v) >> 16);
    return __half_as_ushort(__float2half_rn(v));
}

// Stores the registers K-fastest into an LDS tile [TR][PITCH_H] of 16-bit patterns.
template <bool ROWS_FAST, int HALF, int TR> __device__ __forceinline__ void store_tile_half(const TileRegs<TR> &t, uint32_t *lds) {
#pragma unroll
    for (int h = 0; h < TileRegs<TR>::slots; h++) {
        uint32_t slot = threadIdx.x + h * kThreads;
        if (!ROWS_FAST) {
            uint32_t row = slot / (BK / 4), k = (slot % (BK / 4)) * 4;
            uint2 w;
            w.x = pack_halves<HALF>(t.v[h][0], t.v[h][1]);
            w.y = pack_halves<HALF>(t.v[h][2], t.v[h][3]);
            *reinterpret_cast<uint2 *>(lds + row * PITCH_H + k / 2) = w;
        } else {
            uint32_t row, k;
            rows_fast_slot<TR>(slot, row, k);
            uint16_t *l16 = reinterpret_cast<uint16_t *>(lds);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const uint32_t j = rows_fast_order(slot, i);
                l16[(row + j) * (PITCH_H * 2) + k] = narrow_half<HALF>(pick4(t.v[h], j));
            }
        }
    }
}

// NT / MT: 32-wide MFMA tiles per wave along N / M (the block is 2 x 2 waves).  2: the 128 x 128 macro tile; 4: 256 x 256,
// each wave a 128 x 128 block in 256 accumulation registers, one wave per SIMD: four times the matrix instructions between two
// barriers and half the LDS traffic per flop, for products with enough tiles to fill the chip.
// HALF: 1 / 2: words that are bfloat16 / binary16 values (see above; fp8 values are bfloat16 values too).
// 3 / 4 / 5: operands that are ALREADY narrow in memory — bfloat16 / binary16 / fp8 (E4M3) patterns, k contiguous,
// addressed as 32-bit words of 2 or 4 values (a.K counts words; see pack_operand).  The tiles are loaded and staged as words
// (16-byte loads, K-fastest LDS rows of 32 words + 4, one 128-bit LDS read per fragment); a fragment then is 8 (16) consecutive k of
// a row and feeds one v_mfma_f32_32x32x16_{bf16,f16} (two v_mfma_f32_32x32x16_fp8_fp8): a tile is 64 (128) deep in k, and half (a
// quarter) of the bytes move per flop.
template <bool A_MFAST, bool B_NFAST, int NT, int MT, int HALF>
__global__ __launch_bounds__(kThreads) void mfma_gemm_kernel(const MmArgs a) {
    constexpr int BN = 64 * NT, BM = 64 * MT; // shadow the defaults
    constexpr bool WIDEN = HALF == 1 || HALF == 2; // f32 words narrowed on their way into LDS
    constexpr bool PACKED = HALF >= 3;             // narrow in memory already
    static_assert(!PACKED || (!A_MFAST && !B_NFAST), "packed operands are k-contiguous");
    constexpr int LP = WIDEN ? PITCH_H : PITCH; // words per LDS row
    extern __shared__ float lds_dyn[]; // [2][BM][LP] for A, then [2][BN][LP] for B
    auto lds_a = [&](uint32_t buf) { return lds_dyn + buf * (BM * LP); };
    auto lds_b = [&](uint32_t buf) { return lds_dyn + 2 * BM * LP + buf * (BN * LP); };
    auto stage = [&](const TileRegs<BM> &ta, const TileRegs<BN> &tb, uint32_t buf) {
        if constexpr (WIDEN) {
            store_tile_half<A_MFAST, HALF>(ta, reinterpret_cast<uint32_t *>(lds_a(buf)));
            store_tile_half<B_NFAST, HALF>(tb, reinterpret_cast<uint32_t *>(lds_b(buf)));
        } else {
            store_tile(ta, lds_a(buf));
            store_tile(tb, lds_b(buf));
        }
    };

    // Tile order.  Workgroups are dealt round-robin to the 8 XCDs, each with its own L2, so
    // the linear id is first regrouped to give every XCD one contiguous run of tiles; inside
    // the run tiles advance down a column of kGroupM row-tiles before moving to the next
    // column-tile, so that the tiles in flight on one XCD share A and B panels in its L2
    // instead of each streaming its own from HBM.
    const uint32_t tiles_n = (a.N + BN - 1) / BN, tiles_m = (a.M + BM - 1) / BM;
    const uint32_t ntiles = tiles_m * tiles_n;
    uint32_t lin;
    {
        const uint32_t xcd = blockIdx.x % kXcds, slot = blockIdx.x / kXcds;
        const uint32_t q = ntiles / kXcds, r = ntiles % kXcds;
        lin = xcd * q + (xcd < r ? xcd : r) + slot;
    }
    const uint32_t per_group = kGroupM * tiles_n;
    const uint32_t group = lin / per_group, in_group = lin % per_group;
    const uint32_t first_m = group * kGroupM;
    const uint32_t gsize = (tiles_m - first_m) < kGroupM ? (tiles_m - first_m) : kGroupM;
    const uint32_t tile_m = first_m + in_group % gsize, tile_n = in_group / gsize;
    const uint32_t m0 = tile_m * BM, n0 = tile_n * BN;
    int64_t oa, ob;
    batch_offsets(a, blockIdx.y, oa, ob);
    const uint32_t Kk = a.K;
    const uint32_t *A = a.A + oa, *B = a.B + ob;
    uint32_t *C = a.C + (uint64_t)blockIdx.y * a.M * a.N;

    const uint32_t wave = threadIdx.x / 64, lane = threadIdx.x % 64;
    const uint32_t wm = (wave / 2) * (32 * MT), wn = (wave % 2) * (32 * NT); // wave quadrant
    const uint32_t li = lane % 32, lg = lane / 32;

    float16v acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[i][j][v] = 0.0f;

    TileRegs<BM> ra;
    TileRegs<BN> rb;
    const uint32_t nk = (Kk + BK - 1) / BK;
    load_tile<A_MFAST>(ra, A, a.a_sm, a.a_sk, m0, 0, a.M, Kk, a.a_vec);
    load_tile<B_NFAST>(rb, B, a.b_sn, a.b_sk, n0, 0, a.N, Kk, a.b_vec);
    stage(ra, rb, 0);
    __syncthreads();

    if constexpr (PACKED) {
        // A tile's burst of matrix instructions is an eighth (a sixteenth) as long as the f32 tile's, about as long as a
        // trip to memory: the next tile is staged into the other LDS buffer in the middle of the burst and the loads of
        // the tile after it are asked for right there, a whole burst before they are needed (two sets of tile registers
        // for loads two tiles ahead spill: the accumulators take every accumulation register).
        // a 128-bit fragment is the lane's 8 (fp8: 16) consecutive k of its row: lane group g supplies the second half
        // of each 16-deep step (fp8: bytes 0..7 of both groups form one step, bytes 8..15 the next — A and B agree)
        float4v fa[2][MT], fb[2][NT]; // the fragments of the next 16-deep step are read while the current one multiplies
        int8v fa8[2], fb8[NT];        // fp8: the 32 bytes a lane feeds to one 64-deep instruction; a ring of two A rows, all of B
        // Whole tiles (every tile but a ragged last one) are loaded without a test: a lane's slots sit 32 rows apart at the
        // same k, so its byte offsets into the operands are fixed (rows beyond the edge are clamped: what they contribute
        // lands in accumulator rows that are never stored) and a tile is 16 + 16 loads at a base that moves by one tile.
        uint32_t offa[TileRegs<BM>::slots], offb[TileRegs<BN>::slots];
#pragma unroll
        for (int h = 0; h < TileRegs<BM>::slots; h++) {
            const uint32_t slot = threadIdx.x + h * kThreads, row = min(m0 + slot / (BK / 4), a.M - 1);
            offa[h] = (uint32_t)(((uint64_t)row * (uint64_t)a.a_sm + (slot % (BK / 4)) * 4) * 4);
        }
#pragma unroll
        for (int h = 0; h < TileRegs<BN>::slots; h++) {
            const uint32_t slot = threadIdx.x + h * kThreads, row = min(n0 + slot / (BK / 4), a.N - 1);
            offb[h] = (uint32_t)(((uint64_t)row * (uint64_t)a.b_sn + (slot % (BK / 4)) * 4) * 4);
        }
        const bool lean = (uint64_t)a.M * (uint64_t)a.a_sm < (1ull << 30) && (uint64_t)a.N * (uint64_t)a.b_sn < (1ull << 30); // offsets fit 32 bits
        auto ask = [&](TileRegs<BM> &ta, TileRegs<BN> &tb, uint32_t kt) {
            if (lean && (kt + 1) * BK <= Kk) {
                const char *pa = reinterpret_cast<const char *>(A + (uint64_t)kt * BK), *pb = reinterpret_cast<const char *>(B + (uint64_t)kt * BK);
#pragma unroll
                for (int h = 0; h < TileRegs<BM>::slots; h++) ta.v[h] = *reinterpret_cast<const float4v *>(pa + offa[h]);
#pragma unroll
                for (int h = 0; h < TileRegs<BN>::slots; h++) tb.v[h] = *reinterpret_cast<const float4v *>(pb + offb[h]);
            } else {
                load_tile<false>(ta, A, a.a_sm, a.a_sk, m0, kt * BK, a.M, Kk, a.a_vec);
                load_tile<false>(tb, B, a.b_sn, a.b_sk, n0, kt * BK, a.N, Kk, a.b_vec);
            }
        };
        // One tile: S steps of 16 (fp8: 32) k.  Set 0 holds the fragments of step 0 when a tile begins; every step reads the
        // fragments of the next one while it multiplies.  The barrier stands before the LAST step: by then every wave has
        // read all of this tile's fragments and has staged its share of the next tile into the other buffer, so the first
        // fragments of the next tile are read behind the barrier, under the last step's matrix instructions, and the matrix
        // pipe never drains at a tile border.
        // In the steady state (whole tiles, offsets that fit) the 16 slots of the next tile (one 16-byte LDS store each) and
        // the 16 loads of the tile after it are dealt out between groups of four matrix instructions of the first S - 1 steps:
        // a burst of 16 loads (a KB each) blocks the wave's instruction issue for as long as the texture path takes them.
        constexpr int S = BK / 8;
        auto frag_a = [&](const float *la, const int set, const int kc, const int i) {
            fa[set][i] = *reinterpret_cast<const float4v *>(la + (wm + i * 32 + li) * PITCH + kc * 8 + lg * 4);
        };
        auto frag8 = [&](const float *l, const int d, const uint32_t row0) { // the two fragments of double step d of a row
            const float *p = l + (row0 + li) * PITCH + d * 16 + lg * 4;
            const int4v lo = __builtin_bit_cast(int4v, *reinterpret_cast<const float4v *>(p));
            const int4v hi = __builtin_bit_cast(int4v, *reinterpret_cast<const float4v *>(p + 8));
            return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        };
        auto frag_b = [&](const float *lb, const int set, const int kc, const int j) {
            fb[set][j] = *reinterpret_cast<const float4v *>(lb + (wn + j * 32 + li) * PITCH + kc * 8 + lg * 4);
        };
        auto mma_row = [&](const int set, const int i) {
#pragma unroll
            for (int j = 0; j < NT; j++) {
                if constexpr (HALF == 3) {
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, fa[set][i]),
                                                                        __builtin_bit_cast(bf16x8, fb[set][j]), acc[i][j], 0, 0, 0);
                } else if constexpr (HALF == 4) {
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, fa[set][i]),
                                                                       __builtin_bit_cast(f16x8, fb[set][j]), acc[i][j], 0, 0, 0);
                } else {
                    const long2v pa = __builtin_bit_cast(long2v, fa[set][i]), pb = __builtin_bit_cast(long2v, fb[set][j]);
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_fp8_fp8(pa[0], pb[0], acc[i][j], 0, 0, 0);
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_fp8_fp8(pa[1], pb[1], acc[i][j], 0, 0, 0);
                }
            }
        };
        static_assert(MT == NT && TileRegs<BM>::slots == 8 && TileRegs<BN>::slots == 8, "the slot schedule below is for the 256 x 256 tile");
        auto iteration = [&](const uint32_t kt, auto steady) {
            constexpr bool STEADY = decltype(steady)::value;
            const uint32_t cur = kt & 1;
            const bool next = STEADY || kt + 1 < nk;
            const float *la = lds_a(cur), *lb = lds_b(cur);
            float *na = lds_a(cur ^ 1), *nb = lds_b(cur ^ 1);
            const char *pa = reinterpret_cast<const char *>(A + (uint64_t)(kt + 2) * BK), *pb = reinterpret_cast<const char *>(B + (uint64_t)(kt + 2) * BK);
            auto slot = [&](const int q) { // stage slot q of tile kt + 1, then ask for slot q of tile kt + 2
                const uint32_t sl = threadIdx.x + (q % 8) * kThreads, row = sl / (BK / 4), k = (sl % (BK / 4)) * 4;
                if (q < 8) {
                    *reinterpret_cast<float4v *>(na + row * PITCH + k) = ra.v[q % 8];
                    ra.v[q % 8] = *reinterpret_cast<const float4v *>(pa + offa[q % 8]);
                } else {
                    *reinterpret_cast<float4v *>(nb + row * PITCH + k) = rb.v[q % 8];
                    rb.v[q % 8] = *reinterpret_cast<const float4v *>(pb + offb[q % 8]);
                }
            };
            if constexpr (HALF == 5) {
                // fp8 runs at twice the 16-bit rate only on the 64-deep instruction (v_mfma_scale_f32_32x32x64_f8f6f4 with
                // both scales 2^0; the 16-deep fp8 instruction takes the cycles of the 16-bit one): a lane feeds it 32 bytes
                // of its row, two fragments.  A tile is two such double steps; B's four blocks stay in registers for a double
                // step and are replaced one by one behind the last row's instructions, A rows go through a ring of two.  The
                // barrier stands before the last row of the second double step; 16 slots over the 7 rows before it.
                if constexpr (!STEADY) {
                    // the first and the last tiles: nothing is carried in registers from one tile to the next (the guarded
                    // loads need the registers): stage and ask first, then read this tile's fragments as they are needed
                    if (next) {
                        stage(ra, rb, cur ^ 1);
                        if (kt + 2 < nk) ask(ra, rb, kt + 2);
                    }
                    fa8[0] = frag8(la, 0, wm);
#pragma unroll
                    for (int j = 0; j < NT; j++) fb8[j] = frag8(lb, 0, wn + j * 32);
                }
#pragma unroll
                for (int d = 0; d < 2; d++) {
#pragma unroll
                    for (int i = 0; i < MT; i++) {
                        const bool last = d == 1 && i == MT - 1;
                        if (last) {
                            if constexpr (STEADY) {
                                asm volatile("" ::: "memory");
                                __builtin_amdgcn_s_waitcnt(0xc07f);
                                __builtin_amdgcn_s_barrier();
                                asm volatile("" ::: "memory");
                                fa8[0] = frag8(na, 0, wm);
                            }
                        } else if (i == MT - 1) {
                            fa8[0] = frag8(la, 1, wm);
                        } else {
                            fa8[(i + 1) & 1] = frag8(la, d, wm + (i + 1) * 32);
                        }
#pragma unroll
                        for (int j = 0; j < NT; j++) {
                            acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fa8[i & 1], fb8[j], acc[i][j], 0, 0, 0, 0x7f7f7f7f, 0, 0x7f7f7f7f);
                            if (i == MT - 1) {
                                if (d == 0) fb8[j] = frag8(lb, 1, wn + j * 32);
                                else if constexpr (STEADY) fb8[j] = frag8(nb, 0, wn + j * 32);
                            }
                        }
                        if constexpr (STEADY) {
                            const int g = d * MT + i; // 0..6 before the barrier: 3, 2, 2, 2, 3, 2, 2 slots
                            if (g < 7) {
                                const int first = g < 1 ? 0 : g < 5 ? 3 + (g - 1) * 2 : 12 + (g - 5) * 2;
                                const int count = (g == 0 || g == 4) ? 3 : 2;
#pragma unroll
                                for (int c = 0; c < count; c++) slot(first + c);
                            }
                            __builtin_amdgcn_sched_barrier(0);
                        }
                    }
                }
                if constexpr (!STEADY) __syncthreads();
                return;
            }
#pragma unroll
            for (int kc = 0; kc < S - 1; kc++) {
#pragma unroll
                for (int i = 0; i < MT; i++) {
                    frag_a(la, (kc + 1) & 1, kc + 1, i);
                    frag_b(lb, (kc + 1) & 1, kc + 1, i);
                    mma_row(kc & 1, i);
                    if constexpr (STEADY) {
                        // 16 slots over 12 groups: every third group takes two
                        const int g = kc * MT + i, first = g + (g + 2) / 3;
                        slot(first);
                        if (g % 3 == 0) slot(first + 1);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
                if constexpr (!STEADY) {
                    if (kc == S / 2 - 1 && next) {
                        stage(ra, rb, cur ^ 1);
                        if (kt + 2 < nk) ask(ra, rb, kt + 2);
                    }
                }
            }
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_waitcnt(0xc07f); // lgkmcnt(0): this wave's LDS stores have landed (loads in flight stay in flight)
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
#pragma unroll
            for (int i = 0; i < MT; i++) {
                if (next) {
                    frag_a(na, 0, 0, i);
                    frag_b(nb, 0, 0, i);
                }
                mma_row((S - 1) & 1, i);
                if constexpr (STEADY) __builtin_amdgcn_sched_barrier(0);
            }
        };
        static_assert(S % 2 == 0, "the last step multiplies from set 1 while set 0 is refilled");
        auto first_fragments = [&]() {
            if constexpr (HALF == 5) {
                fa8[0] = frag8(lds_a(0), 0, wm);
#pragma unroll
                for (int j = 0; j < NT; j++) fb8[j] = frag8(lds_b(0), 0, wn + j * 32);
            } else {
#pragma unroll
                for (int i = 0; i < MT; i++) {
                    frag_a(lds_a(0), 0, 0, i);
                    frag_b(lds_b(0), 0, 0, i);
                }
            }
        };
        uint32_t kt = 0;
        if (lean && 3 * BK <= Kk) {
            // tile 1 is asked for slot by slot in the order the loop consumes the slots: only then does the compiler's count
            // of loads in flight at the loop's head match the one at its end, and each LDS store waits for its own load
            // (all but the 15 younger ones) instead of for every load
            const char *pa = reinterpret_cast<const char *>(A + (uint64_t)BK), *pb = reinterpret_cast<const char *>(B + (uint64_t)BK);
#pragma unroll
            for (int h = 0; h < 8; h++) {
                ra.v[h] = *reinterpret_cast<const float4v *>(pa + offa[h]);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int h = 0; h < 8; h++) {
                rb.v[h] = *reinterpret_cast<const float4v *>(pb + offb[h]);
                __builtin_amdgcn_sched_barrier(0);
            }
            first_fragments();
            for (; (kt + 3) * BK <= Kk; kt++) iteration(kt, std::true_type{});
        } else {
            if (nk > 1) ask(ra, rb, 1); // (tile 0 is in LDS buffer 0 by now)
            if constexpr (HALF != 5) first_fragments();
        }
        for (; kt < nk; kt++) iteration(kt, std::false_type{});
    }
    // Operands whose 16-byte loads are legal everywhere (aligned, unit stride along k or along the rows): a lane's slots keep
    // their place in every tile, so its byte offsets into the operands are fixed (rows beyond the edge clamped: their values
    // land in accumulator rows that are never stored) and a whole tile is loaded without a test per slot, at a base that
    // moves by one tile.  (The generic loader's tests and fallbacks cost the 256 x 256 tile 4 % of its time.)
    uint32_t offa_kk[TileRegs<BM>::slots], offb_kk[TileRegs<BN>::slots];
    bool lean_kk = false;
    // (The 256 x 256 tile with both operands row-contiguous, or with one such operand narrowed to bfloat16, has no registers
    // left for the offsets.)
    constexpr bool LEAN = !PACKED && (MT != 4 || (!(A_MFAST && B_NFAST) && !((A_MFAST || B_NFAST) && HALF == 1)));
    if constexpr (LEAN) {
        const bool a_ok = A_MFAST ? (a.a_vec && a.a_sm == 1 && a.M % 4 == 0 && a.M >= 4) : (a.a_vec && a.a_sk == 1 && a.a_sm > 0);
        const bool b_ok = B_NFAST ? (a.b_vec && a.b_sn == 1 && a.N % 4 == 0 && a.N >= 4) : (a.b_vec && a.b_sk == 1 && a.b_sn > 0);
        const uint64_t a_span = A_MFAST ? (uint64_t)Kk * (uint64_t)a.a_sk : (uint64_t)a.M * (uint64_t)a.a_sm;
        const uint64_t b_span = B_NFAST ? (uint64_t)Kk * (uint64_t)a.b_sk : (uint64_t)a.N * (uint64_t)a.b_sn;
        lean_kk = a_ok && b_ok && a.a_sk > 0 && a.b_sk > 0 && a_span < (1ull << 30) && b_span < (1ull << 30); // offsets fit 32 bits
#pragma unroll
        for (int h = 0; h < TileRegs<BM>::slots; h++) {
            const uint32_t slot = threadIdx.x + h * kThreads;
            if constexpr (A_MFAST) {
                uint32_t row, k;
                rows_fast_slot<BM>(slot, row, k);
                offa_kk[h] = (uint32_t)(((uint64_t)k * (uint64_t)a.a_sk + min(m0 + row, a.M - 4)) * 4);
            } else {
                offa_kk[h] = (uint32_t)(((uint64_t)min(m0 + slot / (BK / 4), a.M - 1) * (uint64_t)a.a_sm + (slot % (BK / 4)) * 4) * 4);
            }
        }
#pragma unroll
        for (int h = 0; h < TileRegs<BN>::slots; h++) {
            const uint32_t slot = threadIdx.x + h * kThreads;
            if constexpr (B_NFAST) {
                uint32_t row, k;
                rows_fast_slot<BN>(slot, row, k);
                offb_kk[h] = (uint32_t)(((uint64_t)k * (uint64_t)a.b_sk + min(n0 + row, a.N - 4)) * 4);
            } else {
                offb_kk[h] = (uint32_t)(((uint64_t)min(n0 + slot / (BK / 4), a.N - 1) * (uint64_t)a.b_sn + (slot % (BK / 4)) * 4) * 4);
            }
        }
    }
    auto iterate = [&](const uint32_t kt, auto whole_next) {
        const uint32_t cur = kt & 1;
        const bool more = decltype(whole_next)::value || kt + 1 < nk;
        const float *la = lds_a(cur), *lb = lds_b(cur);
        // While a wave is in its burst of matrix instructions it wins issue arbitration against the other
        // wave of its SIMD (which is loading or storing a tile): the two stop advancing in lock-step and
        // their stalls at the barrier no longer coincide.
        if constexpr (decltype(whole_next)::value) {
            // the next tile is a whole tile of k-contiguous, aligned operands: no test per slot
            const char *pa = reinterpret_cast<const char *>(A + (uint64_t)(kt + 1) * BK * (A_MFAST ? (uint64_t)a.a_sk : 1ull));
            const char *pb = reinterpret_cast<const char *>(B + (uint64_t)(kt + 1) * BK * (B_NFAST ? (uint64_t)a.b_sk : 1ull));
#pragma unroll
            for (int h = 0; h < TileRegs<BM>::slots; h++) ra.v[h] = *reinterpret_cast<const float4v *>(pa + offa_kk[h]);
#pragma unroll
            for (int h = 0; h < TileRegs<BN>::slots; h++) rb.v[h] = *reinterpret_cast<const float4v *>(pb + offb_kk[h]);
        } else if (more) {
            load_tile<A_MFAST>(ra, A, a.a_sm, a.a_sk, m0, (kt + 1) * BK, a.M, Kk, a.a_vec);
            load_tile<B_NFAST>(rb, B, a.b_sn, a.b_sk, n0, (kt + 1) * BK, a.N, Kk, a.b_vec);
        }
        __builtin_amdgcn_s_setprio(1);
        if constexpr (WIDEN) {
            // 16-deep chunks: lane group g supplies k = 16*kc + 8*g .. + 7, one 128-bit LDS read per operand block
#pragma unroll
            for (int kc = 0; kc < BK / 16; kc++) {
                float4v fa[MT], fb[NT];
#pragma unroll
                for (int i = 0; i < MT; i++)
                    fa[i] = *reinterpret_cast<const float4v *>(la + (wm + i * 32 + li) * PITCH_H + kc * 8 + lg * 4);
#pragma unroll
                for (int j = 0; j < NT; j++)
                    fb[j] = *reinterpret_cast<const float4v *>(lb + (wn + j * 32 + li) * PITCH_H + kc * 8 + lg * 4);
#pragma unroll
                for (int i = 0; i < MT; i++)
#pragma unroll
                    for (int j = 0; j < NT; j++) {
                        if constexpr (HALF == 1)
                            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, fa[i]),
                                                                                __builtin_bit_cast(bf16x8, fb[j]), acc[i][j], 0, 0, 0);
                        else
                            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, fa[i]),
                                                                               __builtin_bit_cast(f16x8, fb[j]), acc[i][j], 0, 0, 0);
                    }
            }
        }
        __builtin_amdgcn_s_setprio(0);
        if (more) stage(ra, rb, cur ^ 1);
        __syncthreads();
        };
    {
        uint32_t kt = 0;
        if constexpr (LEAN) {
            if (lean_kk)
                for (; (kt + 2) * BK <= Kk; kt++) iterate(kt, std::true_type{});
        }
        for (; kt < (PACKED ? 0u : nk); kt++) iterate(kt, std::false_type{});
    }

    // D layout of v_mfma_f32_32x32x2_f32: lane (li, lg), register v -> row 8*(v/4) + 4*lg + v%4, col li
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < NT; j++) {
            uint32_t col = n0 + wn + j * 32 + li;
            if (col < a.N) {
#pragma unroll
                for (int v = 0; v < 16; v++) {
                    uint32_t row = m0 + wm + i * 32 + 8 * (v / 4) + 4 * lg + (v % 4);
                    if (row < a.M) C[(uint64_t)row * a.N + col] = asu(acc[i][j][v]);
                }
            }
        }
}

// ------------------------------------------------------------------------------------------
// The 256 x 256 tile of operands that lie narrow in memory, fed by loads that go from memory straight into LDS
// (global_load_lds_dwordx4): no tile registers, no LDS stores, so what a workgroup has in flight is bounded by LDS
// instead of by registers.  The register-staged kernel above keeps one tile step (64 KB) in flight per compute unit
// and a step lasts as long as a trip to memory (about 2 us under load, 31 GB/s per unit, whatever the matrix pipes
// could take); here a step is 64 bytes of k per row (32 values of 16 bits, 64 of fp8), a stage is 32 KB and LDS holds a
// ring of kDldsStages of them: one being multiplied, the others in flight.
// A row's 64 bytes are four 16-byte columns; column c of row r sits at column c ^ ((r >> 2) & 3) of the row's place, so
// that the sixteen lanes that a 128-bit fragment read serves at a time (sixteen consecutive rows, one logical column)
// cover all 64 banks (counted: no bank conflicts; with (r >> 1) & 3, which spreads eight rows over 32 banks, every read
// took two turns).  A load instruction of a wave fills 1 KB = 16 consecutive rows in lane order: lane l fetches row
// l / 4, logical column (l % 4) ^ ((row >> 2) & 3).
// HALF: 3 bfloat16, 4 binary16 (two 16-deep steps per stage), 5 fp8 (one 64-deep step per stage).  a.K counts 32-bit
// words and is a multiple of 64 (whole turns of the ring); rows beyond the edge are clamped as above.
// ------------------------------------------------------------------------------------------
constexpr int kDldsStages = 4;
constexpr uint32_t kDldsOperandBytes = 256 * 64, kDldsStageBytes = 2 * kDldsOperandBytes;
constexpr size_t kDldsLdsBytes = (size_t)kDldsStages * kDldsStageBytes;

template <int HALF, bool NARROW_OUT> __global__ __launch_bounds__(kThreads) void mfma_gemm_dlds_kernel(const MmArgs a) {
    constexpr int NS = kDldsStages;
    static_assert(NS == 4, "the last stages of a tile below are written out for a ring of four");
    extern __shared__ float lds_dyn[];
    typedef __attribute__((address_space(3))) char lds_char;
    lds_char *const lds = (lds_char *)lds_dyn;

    // Tile order as in mfma_gemm_kernel: a run of tiles per XCD, down a column of kGroupM row tiles first.  The grid is one
    // workgroup per compute unit (or per tile if there are fewer); workgroup b takes tiles b, b + grid, b + 2 grid, ...
    const uint32_t tiles_n = a.n_tiles ? a.n_tiles : (a.N + 255) / 256, tiles_m = (a.M + 255) / 256;
    const uint32_t ntiles = tiles_m * tiles_n;
    auto tile_origin = [&](const uint32_t vb, uint32_t &m0, uint32_t &n0) {
        const uint32_t xcd = vb % kXcds, slot = vb / kXcds;
        const uint32_t q = ntiles / kXcds, r = ntiles % kXcds;
        const uint32_t lin = xcd * q + (xcd < r ? xcd : r) + slot;
        const uint32_t per_group = kGroupM * tiles_n;
        const uint32_t group = lin / per_group, in_group = lin % per_group;
        const uint32_t first_m = group * kGroupM;
        const uint32_t gsize = (tiles_m - first_m) < kGroupM ? (tiles_m - first_m) : kGroupM;
        m0 = (first_m + in_group % gsize) * 256;
        n0 = (in_group / gsize) * 256;
    };

    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64;
    const uint32_t wm = (wave / 2) * 128, wn = (wave % 2) * 128;
    const uint32_t li = lane % 32, lg = lane / 32;

    // this lane's share of a stage: instruction q of wave w fills rows 64 w + 16 q .. + 15 of an operand's place
    uint32_t offa[4], offb[4];
    auto set_offa = [&](const uint32_t m0) {
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const uint32_t row = wave * 64 + q * 16 + lane / 4, col = (lane % 4) ^ ((row >> 2) & 3);
            offa[q] = (uint32_t)((uint64_t)min(m0 + row, a.M - 1) * (uint64_t)a.a_sm * 4 + col * 16);
        }
    };
    auto set_offb = [&](const uint32_t n0) {
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const uint32_t row = wave * 64 + q * 16 + lane / 4, col = (lane % 4) ^ ((row >> 2) & 3);
            offb[q] = (uint32_t)((uint64_t)min(n0 + row, a.N - 1) * (uint64_t)a.b_sn * 4 + col * 16);
        }
    };
    const char *const ga = reinterpret_cast<const char *>(a.A), *const gb = reinterpret_cast<const char *>(a.B);
    // load q of stage kt (of the tile whose offsets are set): 0..3 the four of A, 4..7 the four of B
    auto issue = [&](const uint32_t kt, const int q) {
        const char *const p = (q < 4 ? ga : gb) + (uint64_t)kt * 64 + (q < 4 ? offa[q & 3] : offb[q & 3]);
        lds_char *const l = lds + (kt % NS) * kDldsStageBytes + (q < 4 ? 0u : kDldsOperandBytes) + wave * 4096 + (q & 3) * 1024;
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)p, (__attribute__((address_space(3))) void *)l, 16, 0, 0);
    };
    // fragment addresses: row li of a 32-row block, logical column c -> byte li * 64 + ((c ^ sw) * 16)
    const uint32_t sw = (li >> 2) & 3;
    auto frag = [&](const uint32_t stage_base, const uint32_t row0, const uint32_t c) {
        return *reinterpret_cast<const __attribute__((address_space(3))) float4v *>(lds + stage_base + (row0 + li) * 64 + ((c ^ sw) * 16));
    };

    float16v acc[4][4];
    auto clear = [&]() {
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int j = 0; j < 4; j++)
#pragma unroll
                for (int v = 0; v < 16; v++) acc[i][j][v] = 0.0f;
    };
    // D layout of the 32 x 32 instructions: lane (li, lg), register v -> row 8 (v / 4) + 4 lg + v % 4, column li.  A whole
    // tile is stored at a per-lane 32-bit offset from addresses that are the same for every lane (M N < 2^30).
    // With NARROW_OUT the result is rounded to the operands' format here (what the separate rounding pass over the f32 result
    // would give, bit for bit) and stored as its patterns, a quarter or an eighth of the bytes of that f32 result and pass:
    // lanes exchange values so that each stores 32 bits — two columns of one row (16-bit: lanes pair up, the even lane takes
    // the first of two rows, the odd lane the second) or four (fp8: a quad transposes its 4 x 4 values).
    const uint32_t lane_off = ((wm + 4 * lg) * a.N + wn + li) * 4;
    const uint32_t sub = HALF == 5 ? (li & 3) : (li & 1); // this lane's row among the 4 (2) that its group exchanges
    const uint32_t lane_off_narrow = ((wm + 4 * lg + sub) * a.N + wn + li - sub) * (HALF == 5 ? 1 : 2);
    // v_perm_b32 selectors of the quad's transposition (byte values 0..3: the second source's bytes, 4..7: the first's, 12: zero)
    const uint32_t quad_sel_a = (0x0C0C0C0Cu & ~(0xFFu << (8 * sub)) & ~(0xFFu << (8 * ((sub + 1) & 3)))) | (sub << (8 * sub)) | ((4 + sub) << (8 * ((sub + 1) & 3)));
    const uint32_t quad_sel_b = (0x0C0C0C0Cu & ~(0xFFu << (8 * ((sub + 2) & 3))) & ~(0xFFu << (8 * ((sub + 3) & 3)))) | (sub << (8 * ((sub + 2) & 3))) |
                                ((4 + sub) << (8 * ((sub + 3) & 3)));
    auto store = [&](const uint32_t m0, const uint32_t n0) {
        const bool whole = m0 + 256 <= a.M && n0 + 256 <= a.N;
        if (whole && !NARROW_OUT) {
            char *const base = reinterpret_cast<char *>(a.C) + ((uint64_t)m0 * a.N + n0) * 4;
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int j = 0; j < 4; j++) {
#pragma unroll
                    for (int v = 0; v < 16; v++) {
                        const uint32_t r = i * 32 + 8 * (v / 4) + (v % 4);
                        // (written out: the compiler would keep a 64-bit address per row in vector registers)
                        asm volatile("global_store_dword %0, %1, %2" ::"v"(lane_off), "v"(acc[i][j][v]), "s"(base + ((uint64_t)r * a.N + j * 32) * 4) : "memory");
                    }
                    __builtin_amdgcn_sched_barrier(0); // (a block at a time: its 16 values pass through 16 registers)
                }
            return;
        }
        if constexpr (NARROW_OUT) {
            // (N is a multiple of 4: a lane's columns are all inside or all outside; the stores of an edge tile are masked, not made a
            // value at a time, which took longer than the tile: 1500 x 2048 x 8192 on bf16 73 -> 67 us)
            auto rounded = [&](auto whole_) {
                auto inside = [&](const uint32_t r, const int j) {
                    return decltype(whole_)::value || (m0 + wm + 4 * lg + sub + r < a.M && n0 + wn + j * 32 + li - sub < a.N);
                };
                constexpr uint32_t EB = HALF == 5 ? 1 : 2;
                char *const base = reinterpret_cast<char *>(a.C) + ((uint64_t)m0 * a.N + n0) * EB;
#pragma unroll
                for (int i = 0; i < 4; i++)
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        if constexpr (HALF != 5) {
#pragma unroll
                            for (int v = 0; v < 16; v += 2) {
                                // v_cvt_pk_{bf16,f16}_f32 round two values as the rounding pass does (all 2^32 patterns compared)
                                const float2v pair = {acc[i][j][v], acc[i][j][v + 1]};
                                uint32_t mine;
                                if constexpr (HALF == 3) mine = __builtin_bit_cast(uint32_t, __builtin_convertvector(pair, bf16x2));
                                else mine = __builtin_bit_cast(uint32_t, __builtin_convertvector(pair, f16x2));
                                const uint32_t theirs = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)mine, 0xB1, 0xF, 0xF, true); // the pair's other lane
                                // even lane: its and the other's first row; odd lane: the other's and its second row
                                const uint32_t two = __builtin_amdgcn_perm(theirs, mine, sub ? 0x03020706u : 0x05040100u);
                                const uint32_t r = i * 32 + 8 * (v / 4) + (v % 4);
                                if (inside(r, j))
                                    asm volatile("global_store_dword %0, %1, %2" ::"v"(lane_off_narrow), "v"(two), "s"(base + ((uint64_t)r * a.N + j * 32) * 2) : "memory");
                            }
                        } else {
#pragma unroll
                            for (int v = 0; v < 16; v += 4) {
                                // v_cvt_pk_fp8_f32 rounds as the rounding pass does once the magnitude is clamped to 448 (it holds no
                                // infinities) and NaNs are set apart: they become the clamped pattern 0x7e, which the 0x7f below completes
                                // (all 2^32 patterns compared)
                                float xs[4];
                                uint32_t nans = 0;
#pragma unroll
                                for (int k = 0; k < 4; k++) {
                                    const uint32_t u = asu(acc[i][j][v + k]), mag = u & 0x7FFFFFFFu;
                                    xs[k] = asf(min(mag, 0x43E00000u) | (u & 0x80000000u));
                                    nans |= mag > 0x7F800000u ? 0x7Fu << (8 * k) : 0u;
                                }
                                int packed = __builtin_amdgcn_cvt_pk_fp8_f32(xs[0], xs[1], 0, false);
                                packed = __builtin_amdgcn_cvt_pk_fp8_f32(xs[2], xs[3], packed, true);
                                const uint32_t mine = (uint32_t)packed | nans; // byte k: row k of this lane's column
                                // lane q of the quad keeps row q: byte q of every lane's word, at the place of that lane's column
                                const uint32_t r1 = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)mine, 0x39, 0xF, 0xF, true); // of lane q + 1
                                const uint32_t r2 = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)mine, 0x4E, 0xF, 0xF, true); // of lane q + 2
                                const uint32_t r3 = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)mine, 0x93, 0xF, 0xF, true); // of lane q + 3
                                const uint32_t four = __builtin_amdgcn_perm(r1, mine, quad_sel_a) | __builtin_amdgcn_perm(r3, r2, quad_sel_b);
                                const uint32_t r = i * 32 + 8 * (v / 4);
                                if (inside(r, j))
                                    asm volatile("global_store_dword %0, %1, %2" ::"v"(lane_off_narrow), "v"(four), "s"(base + ((uint64_t)r * a.N + j * 32)) : "memory");
                                __builtin_amdgcn_sched_barrier(0);
                            }
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
            };
            if (whole) rounded(std::true_type{});
            else rounded(std::false_type{});
            return;
        }
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const uint32_t col = n0 + wn + j * 32 + li;
                if (col < a.N) {
#pragma unroll
                    for (int v = 0; v < 16; v++) {
                        const uint32_t row = m0 + wm + i * 32 + 8 * (v / 4) + 4 * lg + (v % 4);
                        if (row < a.M) {
                            const uint64_t at = (uint64_t)row * a.N + col;
                            a.C[at] = asu(acc[i][j][v]);
                        }
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
    };

    const uint32_t nk = a.K / 16; // a multiple of NS: stage kt of every tile sits in place kt % NS of the ring
    uint32_t vb = blockIdx.x, m0, n0;
    tile_origin(vb, m0, n0);
    set_offa(m0);
    set_offb(n0);
    // A wave's loads wait for each other in the texture path (a KB each), and while one waits the wave issues nothing:
    // they are dealt out one behind every group of matrix instructions.  The first half of stage kt asks for the second
    // half of the loads (B) of the stage 3 ahead, its second half (behind the barrier, when the place of stage kt is free) for
    // the first half (A) of the stage 4 ahead.  The stages of a workgroup's tiles form one stream: the last four stages of a
    // tile ask for the first stages of the next, and the matrix pipes pause at a tile's end only for the stores of the result.
#pragma unroll
    for (int s = 0; s < NS - 1; s++)
#pragma unroll
        for (int q = 0; q < 8; q++) issue(s, q);
#pragma unroll
    for (int q = 0; q < 4; q++) issue(NS - 1, q);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0f70 | (20 & 15) | ((20 >> 4) << 14)); // vmcnt(20): stage 0 is in LDS
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");

    // wait until at most `stages` younger stages are in flight and every fragment read has returned, then meet the others:
    // the next stage is in LDS for everybody, and nobody reads the current stage's place any more.  (Loads finish in the
    // order asked for; the stores of a finished tile share the counter and only make the wait longer than needed.)
    auto meet = [&](auto stages) {
        constexpr uint32_t n = decltype(stages)::value * 8;
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0x0070 | (n & 15) | ((n >> 4) << 14)); // vmcnt(n) lgkmcnt(0)
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    typedef std::integral_constant<int, 2> Y2;
    typedef std::true_type Ask;

    if constexpr (HALF != 5) {
        float4v fa[2][4], fb[2][4];
        auto mma_row = [&](const int set, const int i) {
#pragma unroll
            for (int j = 0; j < 4; j++) {
                if constexpr (HALF == 3)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, fa[set][i]),
                                                                        __builtin_bit_cast(bf16x8, fb[set][j]), acc[i][j], 0, 0, 0);
                else
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, fa[set][i]),
                                                                       __builtin_bit_cast(f16x8, fb[set][j]), acc[i][j], 0, 0, 0);
            }
        };
        // step c of a stage: lane group g supplies the 8 values of k at 16 c + 8 g: logical column 2 c + g
        auto read = [&](const uint32_t kt, const int set, const int c, const int i) {
            const uint32_t base = (kt % NS) * kDldsStageBytes;
            fa[set][i] = frag(base, wm + i * 32, c * 2 + lg);
            fb[set][i] = frag(base + kDldsOperandBytes, wn + i * 32, c * 2 + lg);
        };
#pragma unroll
        for (int i = 0; i < 4; i++) read(0, 0, 0, i);
        // YOUNGER: stages younger than the next one that may still be in flight when this stage meets the others (-1: the
        // last stage of the last tile); FIRST / SECOND: the loads dealt out in the two halves are those of stages fkt / skt
        auto stage = [&](const uint32_t kt, auto younger, auto first, auto second, const uint32_t fkt, const uint32_t skt) {
            constexpr int YOUNGER = decltype(younger)::value;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                read(kt, 1, 1, i);
                mma_row(0, i);
                if constexpr (decltype(first)::value) issue(fkt, 4 + i);
                __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (YOUNGER >= 0) meet(std::integral_constant<uint32_t, (uint32_t)(YOUNGER < 0 ? 0 : YOUNGER)>{});
#pragma unroll
            for (int i = 0; i < 4; i++) {
                if constexpr (YOUNGER >= 0) read(kt + 1, 0, 0, i);
                mma_row(1, i);
                if constexpr (decltype(second)::value) issue(skt, i);
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        for (;;) {
            // (a workgroup's last tile asks for its own first stages again: one way through the loop, and loads nobody reads)
            const uint32_t nvb = vb + gridDim.x;
            const bool more = nvb < ntiles;
            uint32_t nm0, nn0;
            tile_origin(more ? nvb : vb, nm0, nn0);
            clear();
            uint32_t kt = 0;
            for (; kt + NS < nk; kt++) stage(kt, Y2{}, Ask{}, Ask{}, kt + NS - 1, kt + NS);
            set_offa(nm0);
            stage(kt, Y2{}, Ask{}, Ask{}, kt + NS - 1, 0);
            set_offb(nn0);
            stage(kt + 1, Y2{}, Ask{}, Ask{}, 0, 1);
            stage(kt + 2, Y2{}, Ask{}, Ask{}, 1, 2);
            stage(kt + 3, Y2{}, Ask{}, Ask{}, 2, 3);
            store(m0, n0);
            if (!more) break;
            vb = nvb, m0 = nm0, n0 = nn0;
        }
    } else {
        // fp8: a lane feeds the 64-deep instruction 32 bytes of its row — logical columns g and 2 + g (A and B agree on
        // which bytes of the 64 they are).  The fragments of a stage sit in one of two register sets, the stage's parity;
        // the next stage's are read behind the barrier, under the second half of this stage's instructions.
        int8v fa8[2][4], fb8[2][4];
        auto read8 = [&](const uint32_t kt, const int set, const int i) {
            const uint32_t base = (kt % NS) * kDldsStageBytes;
            const int4v alo = __builtin_bit_cast(int4v, frag(base, wm + i * 32, lg)), ahi = __builtin_bit_cast(int4v, frag(base, wm + i * 32, 2 + lg));
            fa8[set][i] = __builtin_shufflevector(alo, ahi, 0, 1, 2, 3, 4, 5, 6, 7);
            const int4v blo = __builtin_bit_cast(int4v, frag(base + kDldsOperandBytes, wn + i * 32, lg)),
                        bhi = __builtin_bit_cast(int4v, frag(base + kDldsOperandBytes, wn + i * 32, 2 + lg));
            fb8[set][i] = __builtin_shufflevector(blo, bhi, 0, 1, 2, 3, 4, 5, 6, 7);
        };
        auto mma8 = [&](const int set, const int i, const int j) {
            acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fa8[set][i], fb8[set][j], acc[i][j], 0, 0, 0, 0x7f7f7f7f, 0, 0x7f7f7f7f);
        };
#pragma unroll
        for (int i = 0; i < 4; i++) read8(0, 0, i);
        // (a load behind every second matrix instruction, which is twice as long as a 16-bit one)
        auto stage8 = [&](const uint32_t kt, const int set, auto younger, auto first, auto second, const uint32_t fkt, const uint32_t skt) {
            constexpr int YOUNGER = decltype(younger)::value;
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    mma8(set, i, 2 * h);
                    mma8(set, i, 2 * h + 1);
                    if constexpr (decltype(first)::value) issue(fkt, 4 + 2 * i + h);
                    __builtin_amdgcn_sched_barrier(0);
                }
            if constexpr (YOUNGER >= 0) meet(std::integral_constant<uint32_t, (uint32_t)(YOUNGER < 0 ? 0 : YOUNGER)>{});
#pragma unroll
            for (int i = 2; i < 4; i++)
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    if constexpr (YOUNGER >= 0) read8(kt + 1, set ^ 1, 2 * (i - 2) + h);
                    mma8(set, i, 2 * h);
                    mma8(set, i, 2 * h + 1);
                    if constexpr (decltype(second)::value) issue(skt, 2 * (i - 2) + h);
                    __builtin_amdgcn_sched_barrier(0);
                }
        };
        for (;;) {
            const uint32_t nvb = vb + gridDim.x;
            const bool more = nvb < ntiles;
            uint32_t nm0, nn0;
            tile_origin(more ? nvb : vb, nm0, nn0);
            clear();
            uint32_t kt = 0;
            for (; kt + NS < nk; kt += 2) {
                stage8(kt, 0, Y2{}, Ask{}, Ask{}, kt + NS - 1, kt + NS);
                stage8(kt + 1, 1, Y2{}, Ask{}, Ask{}, kt + NS, kt + NS + 1);
            }
            set_offa(nm0);
            stage8(kt, 0, Y2{}, Ask{}, Ask{}, kt + NS - 1, 0);
            set_offb(nn0);
            stage8(kt + 1, 1, Y2{}, Ask{}, Ask{}, 0, 1);
            stage8(kt + 2, 0, Y2{}, Ask{}, Ask{}, 1, 2);
            stage8(kt + 3, 1, Y2{}, Ask{}, Ask{}, 2, 3);
            store(m0, n0);
            if (!more) break;
            vb = nvb, m0 = nm0, n0 = nn0;
        }
    }
    // (loads into LDS must not outlive the workgroup: its LDS passes to the next one)
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0070); // vmcnt(0) lgkmcnt(0)
}

// ------------------------------------------------------------------------------------------
// Skinny kernel: M <= 8, B rows K-contiguous (b_sk == 1).  One wave per output column.
// ------------------------------------------------------------------------------------------
template <int MM> __global__ __launch_bounds__(kThreads) void skinny_kt_kernel(const MmArgs a) {
    const uint32_t wave = threadIdx.x / 64, lane = threadIdx.x % 64;
    const uint32_t n = blockIdx.x * (kThreads / 64) + wave;
    if (n >= a.N) return;
    int64_t oa, ob;
    batch_offsets(a, blockIdx.y, oa, ob);
    const uint32_t *A = a.A + oa;
    const uint32_t *Brow = a.B + ob + (int64_t)n * a.b_sn;
    float acc[MM];
#pragma unroll
    for (int m = 0; m < MM; m++) acc[m] = 0.0f;
    const bool vec = a.b_vec && a.a_vec && a.a_sk == 1 && (a.K % 4 == 0);
    if (vec) {
        for (uint32_t k = lane * 4; k < a.K; k += 256) {
            float4v b = *reinterpret_cast<const float4v *>(Brow + k);
#pragma unroll
            for (int m = 0; m < MM; m++) {
                if ((uint32_t)m < a.M) {
                    float4v x = *reinterpret_cast<const float4v *>(A + (int64_t)m * a.a_sm + k);
                    acc[m] = fmaf(x[0], b[0], acc[m]);
                    acc[m] = fmaf(x[1], b[1], acc[m]);
                    acc[m] = fmaf(x[2], b[2], acc[m]);
                    acc[m] = fmaf(x[3], b[3], acc[m]);
                }
            }
        }
    } else {
        for (uint32_t k = lane; k < a.K; k += 64) {
            float b = asf(Brow[k]);
#pragma unroll
            for (int m = 0; m < MM; m++)
                if ((uint32_t)m < a.M) acc[m] = fmaf(asf(A[(int64_t)m * a.a_sm + (int64_t)k * a.a_sk]), b, acc[m]);
        }
    }
#pragma unroll
    for (int m = 0; m < MM; m++) {
        const float v = wave_add<1>(acc[m]);
        if (lane == 0 && (uint32_t)m < a.M) a.C[((uint64_t)blockIdx.y * a.M + m) * a.N + n] = asu(v);
    }
}


// Vectorised skinny kernel for K > 256: a wave owns COLS output columns and walks K with
// 16-byte loads (COLS weight loads + M activation loads in flight per lane per trip; the
// activation rows stay in L1/L2).  SPLIT: the four waves of the block share the columns
// and split K, for shapes with too few columns to fill the chip.
#ifndef CG_WIDE_UNROLL
#define CG_WIDE_UNROLL 2
#endif
template <int MM, int COLS, bool SPLIT>
__device__ __forceinline__ void skinny_kt_wide_body(const MmArgs &a, const uint32_t block_x, const uint32_t block_y) {
    constexpr int kWideUnroll = COLS == 1 ? CG_WIDE_UNROLL : 2;
    const uint32_t wave = threadIdx.x / 64, lane = threadIdx.x % 64;
    const uint32_t group = SPLIT ? block_x : block_x * 4 + wave;
    const uint32_t n0 = group * COLS;
    const bool live = n0 < a.N;
    int64_t oa, ob;
    batch_offsets(a, block_y, oa, ob);
    const uint32_t *A = a.A + oa;
    const uint32_t *B = a.B + ob;
    float acc[COLS][MM];
#pragma unroll
    for (int c = 0; c < COLS; c++)
#pragma unroll
        for (int m = 0; m < MM; m++) acc[c][m] = 0.0f;
    if (live) {
        const uint32_t kstep = SPLIT ? 1024u : 256u;
#pragma unroll kWideUnroll
        for (uint32_t k = (SPLIT ? wave * 256u : 0u) + lane * 4; k < a.K; k += kstep) {
            float4v w[COLS], x[MM];
#pragma unroll
            for (int c = 0; c < COLS; c++) {
                w[c] = (float4v){0.f, 0.f, 0.f, 0.f};
                if (n0 + c < a.N) w[c] = *reinterpret_cast<const float4v *>(B + (int64_t)(n0 + c) * a.b_sn + k);
            }
#pragma unroll
            for (int m = 0; m < MM; m++) {
                x[m] = (float4v){0.f, 0.f, 0.f, 0.f};
                if ((uint32_t)m < a.M) x[m] = *reinterpret_cast<const float4v *>(A + (int64_t)m * a.a_sm + k);
            }
#pragma unroll
            for (int c = 0; c < COLS; c++)
#pragma unroll
                for (int m = 0; m < MM; m++) {
                    acc[c][m] = fmaf(x[m][0], w[c][0], acc[c][m]);
                    acc[c][m] = fmaf(x[m][1], w[c][1], acc[c][m]);
                    acc[c][m] = fmaf(x[m][2], w[c][2], acc[c][m]);
                    acc[c][m] = fmaf(x[m][3], w[c][3], acc[c][m]);
                }
        }
    }
#pragma unroll
    for (int c = 0; c < COLS; c++)
#pragma unroll
        for (int m = 0; m < MM; m++) acc[c][m] = wave_add<1>(acc[c][m]);
    if (SPLIT) {
        __shared__ float part[4][COLS * MM];
        if (lane == 0) {
#pragma unroll
            for (int c = 0; c < COLS; c++)
#pragma unroll
                for (int m = 0; m < MM; m++) part[wave][c * MM + m] = acc[c][m];
        }
        __syncthreads();
        if (threadIdx.x < COLS * MM) {
            uint32_t c = threadIdx.x / MM, m = threadIdx.x % MM;
            float v = (part[0][threadIdx.x] + part[1][threadIdx.x]) + (part[2][threadIdx.x] + part[3][threadIdx.x]);
            if (n0 + c < a.N && m < a.M) a.C[((uint64_t)block_y * a.M + m) * a.N + n0 + c] = asu(v);
        }
    } else if (live && lane == 0) {
#pragma unroll
        for (int c = 0; c < COLS; c++)
#pragma unroll
            for (int m = 0; m < MM; m++)
                if (n0 + c < a.N && (uint32_t)m < a.M) a.C[((uint64_t)block_y * a.M + m) * a.N + n0 + c] = asu(acc[c][m]);
    }
}

template <int MM, int COLS, bool SPLIT>
__global__ __launch_bounds__(kThreads) void skinny_kt_wide_kernel(const MmArgs a) {
    skinny_kt_wide_body<MM, COLS, SPLIT>(a, blockIdx.x, blockIdx.y);
}

// Chunks of 2048 values of k when K is a multiple of that, of 1024 when of that (hidden sizes like 1024 or 3072); any
// other K (a multiple of 4 above 256: hidden sizes like 576 or 1536) runs with a ragged last chunk, the waves of a
// workgroup then interleaved every 64 values of k (xreg_lane_k) so that a short chunk still spreads over all four.
static inline int xreg_trips(uint32_t K) {
    return K % 2048 == 0 ? 8 : K % 1024 == 0 ? 4 : (K % 4 == 0 && K > 256) ? (K > 1024 ? 8 : 4) : 0;
}
// Column groups per workgroup of the packed kernel: as many as leave about two workgroups per compute unit
// (env CG_XREG_ITERS=n forces n, for measurements).
static inline uint32_t xreg_cols_iters(uint64_t groups) {
    static const int forced = [] {
        const char *e = getenv("CG_XREG_ITERS");
        return e ? atoi(e) : 0;
    }();
    if (forced > 0) return (uint32_t)forced;
    const uint64_t it = groups / 512;
    return (uint32_t)(it < 1 ? 1 : it > 4 ? 4 : it);
}
// Five to eight rows: a second group of four.
static inline bool xreg_narrow(uint32_t M, uint32_t K) { return M >= 1 && M <= 8 && xreg_trips(K) != 0; }
// Skinny kernel on the 4x4x1 matrix instruction (16 independent 4x4 outer products per
// issue): lane (b, j) = (lane / 4, lane % 4) feeds weight W[n0 + j][k] and activation
// X[j][k] for the k values of block b, so one 16-byte weight load per lane drives four
// instructions that update all 4 (rows) x 4 (columns) partial sums of the block.  Against
// the FMA kernels this needs a quarter of the vector issue slots.  The four waves of a
// workgroup split each 2048-wide chunk of k into runs of 512, keep their share of the chunk's activations in registers (8 x 16 bytes
// per lane and row group) and reuse it for CG groups of four columns, so the activation rows
// are fetched once per 4 * CG columns.
//
// Where a lane's k values lie inside a chunk of TRIPS * 256: trip t covers k0 + kb + ks * t .. + 3.  Whole chunks: a wave
// takes a quarter of the chunk in a row (2 KiB in a row of each weight row: measured 12 % faster on the gate / up pair than
// interleaving the waves every 256 bytes).  A ragged last chunk: the waves interleaved every 64 values of k, so that what
// there is of the chunk is shared by all four.
// WHOLE: K is whole chunks (a kernel of its own: the registers of the other's branches would cost a workgroup per compute unit).
template <int TRIPS, bool WHOLE> __device__ __forceinline__ void xreg_lane_k(uint32_t wave, uint32_t b, uint32_t &kb, uint32_t &ks) {
    kb = (WHOLE ? wave * (TRIPS * 64) : wave * 64) + b * 4;
    ks = WHOLE ? 64u : 256u;
}
template <class F> static void xreg_either(uint32_t K, int trips, F f) { // f(is K whole chunks of that many trips, as a constant)
    if (trips && K % (trips * 256) == 0) f(std::true_type{});
    else f(std::false_type{});
}
// A chunk's work with as many trips as what is left of K has (or one more): f(their number, as a constant).  Trips that lie behind K
// altogether would be asked for like any others, clamped: 4 x 2308 x 12288 24.7 us with all of a chunk's trips, 19.1 so.
template <int TRIPS, bool WHOLE, class F> __device__ __forceinline__ void xreg_chunk(uint32_t left, F f) {
    static_assert(TRIPS == 8 || TRIPS == 4, "chunks of 2048 or 1024");
    constexpr std::integral_constant<int, TRIPS> all{};
    if constexpr (WHOLE) {
        f(all);
    } else if constexpr (TRIPS == 8) {
        if (left > 6 * 256) f(all);
        else if (left > 4 * 256) f(std::integral_constant<int, 6>{});
        else if (left > 3 * 256) f(std::integral_constant<int, 4>{});
        else if (left > 2 * 256) f(std::integral_constant<int, 3>{});
        else f(std::integral_constant<int, 2>{});
    } else {
        if (left > 3 * 256) f(all);
        else if (left > 2 * 256) f(std::integral_constant<int, 3>{});
        else f(std::integral_constant<int, 2>{});
    }
}
// Four values of a row from k on, and what they count for: zeros behind K.  Loads behind K are clamped, not tested: a test in front of
// every load leaves the compiler without a count of what is on its way, and it then waits for all of it before each of several groups.
// The kernel below runs for a few microseconds, most of them one trip to memory; around it nothing waits that need not: every load of
// a chunk is on its way before the first wait, and the sums over lanes stay out of LDS (four_sums).
template <bool WHOLE> __device__ __forceinline__ float4v xreg_at(const uint32_t *row, uint32_t k, uint32_t K) {
    return *reinterpret_cast<const float4v *>(row + (WHOLE ? k : min(k, K - 4)));
}
template <bool WHOLE> __device__ __forceinline__ float4v xreg_within(float4v v, uint32_t k, uint32_t K) {
    if constexpr (!WHOLE) {
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = k < K ? v[e] : 0.0f;
    }
    return v;
}
template <bool WHOLE, int MM, int CG, int TRIPS> __global__ __launch_bounds__(kThreads) void skinny_kt_mfma_xreg_kernel(const MmArgs a) {
    static_assert(MM == 4 || MM == 8, "one or two groups of four rows");
    constexpr int G = MM / 4;
    const uint32_t wave = threadIdx.x / 64, lane = threadIdx.x % 64;
    const uint32_t j = lane % 4, b = lane / 4;
    const uint32_t n0 = blockIdx.x * (4 * CG);
    int64_t oa, ob;
    batch_offsets(a, blockIdx.y, oa, ob);
    const uint32_t *wrow[CG];
#pragma unroll
    for (int c = 0; c < CG; c++) wrow[c] = a.B + ob + (int64_t)min(n0 + 4 * c + j, a.N - 1) * a.b_sn;
    const uint32_t *xrow[G];
#pragma unroll
    for (int g = 0; g < G; g++) xrow[g] = a.A + oa + (int64_t)min((uint32_t)(4 * g) + j, a.M - 1) * a.a_sm;
    float4v acc[CG][G];
#pragma unroll
    for (int c = 0; c < CG; c++)
#pragma unroll
        for (int g = 0; g < G; g++) acc[c][g] = (float4v){0.f, 0.f, 0.f, 0.f};
    // of every chunk of TRIPS * 256 values of k (2048 or 1024) a wave takes a quarter in a row (TRIPS trips of 64)
    uint32_t kb, ks;
    xreg_lane_k<TRIPS, WHOLE>(wave, b, kb, ks);
    uint32_t k0 = 0;
    auto chunk = [&](auto trips) __attribute__((always_inline)) {
        constexpr int T = decltype(trips)::value;
        float4v xr[G][T];
#pragma unroll
        for (int t = 0; t < T; t++)
#pragma unroll
            for (int g = 0; g < G; g++) xr[g][t] = xreg_at<WHOLE>(xrow[g], k0 + kb + ks * t, a.K);
#pragma unroll
        for (int c = 0; c < CG; c++) {
            float4v w[T];
#pragma unroll
            for (int t = 0; t < T; t++) w[t] = xreg_at<WHOLE>(wrow[c], k0 + kb + ks * t, a.K);
            if constexpr (!WHOLE) __builtin_amdgcn_sched_barrier(0); // (what follows stays behind all of the loads)
            if constexpr (!WHOLE) {
#pragma unroll
                for (int t = 0; t < T; t++) {
                    w[t] = xreg_within<WHOLE>(w[t], k0 + kb + ks * t, a.K);
#pragma unroll
                    for (int g = 0; g < G; g++)
                        if (c == 0) xr[g][t] = xreg_within<WHOLE>(xr[g][t], k0 + kb + ks * t, a.K);
                }
            }
#pragma unroll
            for (int t = 0; t < T; t++)
#pragma unroll
                for (int g = 0; g < G; g++)
#pragma unroll
                    for (int e = 0; e < 4; e++) acc[c][g] = __builtin_amdgcn_mfma_f32_4x4x1f32(xr[g][t][e], w[t][e], acc[c][g], 0, 0, 0);
        }
    };
    for (; k0 < a.K; k0 += TRIPS * 256) xreg_chunk<TRIPS, WHOLE>(a.K - k0, chunk);
    __shared__ float part[4][CG * MM * 4];
#pragma unroll
    for (int c = 0; c < CG; c++)
#pragma unroll
        for (int g = 0; g < G; g++) {
            const float v = four_sums(acc[c][g][0], acc[c][g][1], acc[c][g][2], acc[c][g][3]); // of row g * 4 + b / 4
            if (b % 4 == 0) part[wave][(c * MM + 4 * g) * 4 + b + j] = v;
        }
    __syncthreads();
    if (threadIdx.x < CG * MM * 4) {
        const uint32_t c = threadIdx.x / (MM * 4), m = threadIdx.x / 4 % MM, col = n0 + 4 * c + threadIdx.x % 4;
        const uint32_t v = asu((part[0][threadIdx.x] + part[1][threadIdx.x]) + (part[2][threadIdx.x] + part[3][threadIdx.x]));
        if (col < a.N && m < a.M) a.C[((uint64_t)blockIdx.y * a.M + m) * a.N + col] = v;
    }
}

// The store above for products whose heads go through an RMS norm of their own first (RopeStore::hgamma, the q / k norm of
// Qwen3): the norm needs the sum of squares over all hd columns of a head, which lie with several workgroups of the
// products' kernel, and workgroups cannot exchange values inside a launch for less than a launch costs.
// So that kernel leaves those products plain (rows already divided by the input norm) in scratch memory, N columns a row.  Decode-time
// attention finishes them as it loads them (see OpenHeads); where something else comes first or the attention is none of those kernels',
// this small launch does: a workgroup per head of a product, a thread per (row, column) of the head; the
// head's norm, the embedding and the store, op for op as the stand-alone programs but for norm_divisor's square root and the order of the
// sum of squares (in runs of 16 columns).  A thread norms its partner of the embedding as well, so that all loads go together and one barrier is enough: 4.8 -> 3.0 us for 24 heads
// of 128 (3.5 in the steps of the Qwen3-0.6B shape, 16 and 8 heads).  Measured against one launch with a
// workgroup of 1024 threads per head (a compute unit streams about 25 GB/s on its own however deep its loads are queued,
// so that launch is as slow as its heads are few: 23 to 29 us for the 32 heads of 128 x 1024 of the Qwen3-0.6B shape):
// 9 + 3 us and a hand-over, 1.94 -> 1.66 ms per decode step of that shape.
struct HeadFinish {
    RopeStore s[kMaxSkinny];
    const uint32_t *src[kMaxSkinny];
    uint32_t N[kMaxSkinny];
    uint32_t n, M;
};
constexpr int kFinishThreads = 1024;
__global__ __launch_bounds__(kFinishThreads) void head_norm_rope_finish_kernel(const HeadFinish f) {
    const uint32_t p = blockIdx.y, head = blockIdx.x, hd = f.s[p].hd, N = f.N[p];
    if (head * hd >= N) return;
    const RopeStore &rs = f.s[p];
    const uint32_t e = threadIdx.x, m = e / hd, d = e - m * hd;
    const bool mine = e < f.M * hd; // (M <= 8, hd <= 128: at most 1024 threads)
    // the value and the one that the embedding mixes it with: lower half -x[d + hd / 2], upper half x[d - hd / 2]
    const bool low = d < hd / 2;
    const uint32_t d2 = rs.rope ? (low ? d + hd / 2 : d - hd / 2) : d;
    uint32_t v = 0, v2 = 0, hg = 0, hg2 = 0, cs = 0, sn = 0;
    if (mine) { // (all loads together)
        const uint32_t *const row = f.src[p] + (int64_t)m * N + head * hd;
        v = row[d];
        v2 = row[d2];
        hg = rs.hgamma[d];
        hg2 = rs.hgamma[d2];
        if (rs.rope) {
            cs = rs.cos[d];
            sn = rs.sin[d];
        }
    }
    // the row's sum of squares: 16 columns by their lanes (head sizes are multiples of 16), then run after run
    __shared__ float runs[kFinishThreads / 16];
    float ss = mine ? asf(v) * asf(v) : 0.0f;
    ss = asf(group_fold<16>(asu(ss), AddWords{}));
    if (e % 16 == 0) runs[e / 16] = ss;
    __syncthreads();
    if (!mine) return;
    ss = 0.0f;
    for (uint32_t c = 0; c < hd / 16; c++) ss += runs[m * (hd / 16) + c];
    const uint32_t r = asu(norm_divisor(ss, rs.hn_n_bits, rs.hn_eps_bits, rs.hn_exp_bits));
    v = apply<kMul, true>(apply<kDiv, true>(v, r, 0, nullptr), hg, 0, nullptr);
    if (rs.rope) {
        const uint32_t other = apply<kMul, true>(apply<kDiv, true>(v2, r, 0, nullptr), hg2, 0, nullptr);
        const uint32_t rot = low ? apply<kNeg, true>(other, 0, 0, nullptr) : other;
        v = apply<kAdd, true>(apply<kMul, true>(cs, v, 0, nullptr), apply<kMul, true>(sn, rot, 0, nullptr), 0, nullptr);
    }
    rs.dst[(int64_t)m * rs.sb + (int64_t)head * rs.sh + d] = v;
}

// Vectorised skinny kernel for short K (K <= 4*LPC, e.g. q.K^T of a decode step with
// K = head_dim): LPC lanes share a column, so a wave covers 64/LPC columns per pass and
// the activation fragment is loaded once.
template <int MM, int LPC> __global__ __launch_bounds__(kThreads) void skinny_kt_narrow_kernel(const MmArgs a) {
    constexpr uint32_t CPW = 64 / LPC, PASSES = 4;
    const uint32_t wave = threadIdx.x / 64, lane = threadIdx.x % 64;
    const uint32_t sub = lane / LPC, l = lane % LPC;
    const uint32_t nblock = blockIdx.x * (4 * CPW * PASSES);
    int64_t oa, ob;
    batch_offsets(a, blockIdx.y, oa, ob);
    const uint32_t *A = a.A + oa;
    const uint32_t *B = a.B + ob;
    const uint32_t k = l * 4;
    const bool kin = k < a.K;
    float4v x[MM];
#pragma unroll
    for (int m = 0; m < MM; m++) {
        x[m] = (float4v){0.f, 0.f, 0.f, 0.f};
        if (kin && (uint32_t)m < a.M) x[m] = *reinterpret_cast<const float4v *>(A + (int64_t)m * a.a_sm + k);
    }
    float4v w[PASSES];
#pragma unroll
    for (uint32_t p = 0; p < PASSES; p++) {
        uint32_t col = nblock + (p * 4 + wave) * CPW + sub;
        w[p] = (float4v){0.f, 0.f, 0.f, 0.f};
        if (kin && col < a.N) w[p] = *reinterpret_cast<const float4v *>(B + (int64_t)col * a.b_sn + k);
    }
#pragma unroll
    for (uint32_t p = 0; p < PASSES; p++) {
        uint32_t col = nblock + (p * 4 + wave) * CPW + sub;
#pragma unroll
        for (int m = 0; m < MM; m++) {
            float v = fmaf(x[m][3], w[p][3], fmaf(x[m][2], w[p][2], fmaf(x[m][1], w[p][1], x[m][0] * w[p][0])));
#pragma unroll
            for (int s = LPC / 2; s >= 1; s >>= 1) v += __shfl_xor(v, s);
            if (l == 0 && col < a.N && (uint32_t)m < a.M) a.C[((uint64_t)blockIdx.y * a.M + m) * a.N + col] = asu(v);
        }
    }
}

// Skinny kernel for N-contiguous B (p.V of a decode step: M = 1, K = T, N = head_dim):
// a block owns 64 output columns (16 lanes x float4) and splits K over 16 lane groups,
// which an LDS exchange sums at the end.
template <int MM>
__global__ __launch_bounds__(kThreads) void skinny_nn_kernel(const MmArgs a, uint32_t *dst, uint32_t kchunk) {
    const uint32_t ng = threadIdx.x % 16, kg = threadIdx.x / 16;
    const uint32_t n = blockIdx.x * 64 + ng * 4;
    int64_t oa, ob;
    batch_offsets(a, blockIdx.y, oa, ob);
    const uint32_t *A = a.A + oa;
    const uint32_t *B = a.B + ob;
    float4v acc[MM];
#pragma unroll
    for (int m = 0; m < MM; m++) acc[m] = (float4v){0.f, 0.f, 0.f, 0.f};
    const bool vec = a.b_vec && n + 3 < a.N;
    const uint32_t kbeg = blockIdx.z * kchunk, kend = min(a.K, kbeg + kchunk);
#pragma unroll 4
    for (uint32_t k = kbeg + kg; k < kend; k += 16) {
        const uint32_t *p = B + (int64_t)k * a.b_sk + (int64_t)n * a.b_sn;
        float4v w;
        if (vec) {
            w = *reinterpret_cast<const float4v *>(p);
        } else {
            w[0] = ld_guard(p, n < a.N);
            w[1] = ld_guard(p + a.b_sn, n + 1 < a.N);
            w[2] = ld_guard(p + 2 * a.b_sn, n + 2 < a.N);
            w[3] = ld_guard(p + 3 * a.b_sn, n + 3 < a.N);
        }
#pragma unroll
        for (int m = 0; m < MM; m++) {
            if ((uint32_t)m < a.M) {
                float x = asf(A[(int64_t)m * a.a_sm + (int64_t)k * a.a_sk]);
                acc[m][0] = fmaf(x, w[0], acc[m][0]);
                acc[m][1] = fmaf(x, w[1], acc[m][1]);
                acc[m][2] = fmaf(x, w[2], acc[m][2]);
                acc[m][3] = fmaf(x, w[3], acc[m][3]);
            }
        }
    }
    __shared__ float red[16][64 * MM + 4];
#pragma unroll
    for (int m = 0; m < MM; m++)
#pragma unroll
        for (int j = 0; j < 4; j++) red[kg][m * 64 + ng * 4 + j] = acc[m][j];
    __syncthreads();
    for (uint32_t o = threadIdx.x; o < 64 * MM; o += kThreads) {
        float v = 0.0f;
#pragma unroll
        for (int g = 0; g < 16; g++) v += red[g][o];
        uint32_t m = o / 64, col = blockIdx.x * 64 + o % 64;
        // dst is C itself (gridDim.z == 1) or the [batch][gridDim.z][M][N] partial sums
        if (m < a.M && col < a.N)
            dst[(((uint64_t)blockIdx.y * gridDim.z + blockIdx.z) * a.M + m) * a.N + col] = asu(v);
    }
}

// C[b][e] = sum over s of part[b][s][e]   (e < M*N), in a fixed order
__global__ __launch_bounds__(kThreads) void splitk_reduce_kernel(const uint32_t *part, uint32_t *C, uint32_t splits,
                                                                 uint32_t mn, uint64_t total) {
    uint64_t i = (uint64_t)blockIdx.x * kThreads + threadIdx.x;
    if (i >= total) return;
    uint64_t b = i / mn, e = i % mn;
    float v = 0.0f;
    for (uint32_t s = 0; s < splits; s++) v += asf(part[(b * splits + s) * mn + e]);
    C[i] = asu(v);
}

// ------------------------------------------------------------------------------------------
// Plain kernel: one thread per output element.  u32 with wrapping arithmetic
// (ndarray.rs:181) and the f32 shapes nothing else takes.
// ------------------------------------------------------------------------------------------
template <bool F> __global__ __launch_bounds__(kThreads) void simple_gemm_kernel(const MmArgs a) {
    uint64_t e = (uint64_t)blockIdx.x * kThreads + threadIdx.x;
    if (e >= (uint64_t)a.M * a.N) return;
    uint32_t m = (uint32_t)(e / a.N), n = (uint32_t)(e % a.N);
    int64_t oa, ob;
    batch_offsets(a, blockIdx.y, oa, ob);
    const uint32_t *A = a.A + oa + (int64_t)m * a.a_sm;
    const uint32_t *B = a.B + ob + (int64_t)n * a.b_sn;
    uint32_t r;
    if (F) {
        float s = 0.0f;
        for (uint32_t k = 0; k < a.K; k++) s = fmaf(asf(A[(int64_t)k * a.a_sk]), asf(B[(int64_t)k * a.b_sk]), s);
        r = asu(s);
    } else {
        uint32_t s = 0;
        for (uint32_t k = 0; k < a.K; k++) s += A[(int64_t)k * a.a_sk] * B[(int64_t)k * a.b_sk];
        r = s;
    }
    a.C[(uint64_t)blockIdx.y * a.M * a.N + e] = r;
}

} // namespace

int fold_matmul(const cg_tensor *x, const cg_tensor *y, MmFold *f) {
    const int r = x->rank;
    int64_t M = x->dims[r - 2];
    auto stride = [](const cg_tensor *t, int ax) -> int64_t { return t->uniform ? 0 : t->strides[ax]; };
    f->a_sm = stride(x, r - 2);
    f->a_sk = stride(x, r - 1);
    f->b_sk = stride(y, r - 2);
    f->b_sn = stride(y, r - 1);
    // collapse the batch axes of A and B together (C is row-major, so it follows); a split axis of
    // either operand contributes its two parts as separate axes
    int64_t bd[kMaxRank + 1], sa[kMaxRank + 1], sb[kMaxRank + 1];
    int w = 0;
    auto push_axis = [&](int64_t d, int64_t s1, int64_t s2) {
        if (d == 1) return;
        if (w > 0 && sa[w - 1] == s1 * d && sb[w - 1] == s2 * d) {
            bd[w - 1] *= d;
            sa[w - 1] = s1;
            sb[w - 1] = s2;
        } else {
            bd[w] = d;
            sa[w] = s1;
            sb[w] = s2;
            w++;
        }
    };
    for (int i = 0; i < r - 2; i++) {
        const int64_t d = x->dims[i], s1 = stride(x, i), s2 = stride(y, i);
        const bool xs = x->split == i, ys = y->split == i;
        if (xs || ys) {
            const int64_t inner = xs ? x->split_inner : y->split_inner;
            push_axis(d / inner, xs ? x->split_os : s1 * inner, ys ? y->split_os : s2 * inner);
            push_axis(inner, s1, s2);
        } else {
            push_axis(d, s1, s2);
        }
    }
    // fold the innermost batch axis into M when B ignores it and A walks it as more rows
    while (w > 0 && sb[w - 1] == 0 && (M == 1 || sa[w - 1] == f->a_sm * M)) {
        if (M == 1) f->a_sm = sa[w - 1];
        M *= bd[w - 1];
        w--;
    }
    if (w > kMaxBatchAxes) return fail(CG_ERR_UNSUPPORTED, "matmul: more than %d non-mergeable batch axes", kMaxBatchAxes);
    int64_t batch = 1;
    for (int i = 0; i < w; i++) batch *= bd[i];
    f->M = M;
    f->N = y->dims[r - 1];
    f->K = x->dims[r - 1];
    f->batch = batch;
    f->nb = w;
    for (int d = 0; d < w; d++) {
        f->bd[d] = bd[w - 1 - d];
        f->a_bs[d] = sa[w - 1 - d];
        f->b_bs[d] = sb[w - 1 - d];
    }
    return CG_OK;
}

// Kernel arguments of x . y -> c (row-major); the folded extents come back in *f.
// The geometry of x . y (everything of MmArgs but the operands' addresses and what depends on them).
static int mm_geometry(const cg_tensor *x, const cg_tensor *y, void *c, MmArgs *ap, MmFold *fp) {
    MmArgs &a = *ap;
    memset(&a, 0, sizeof a);
    a.C = static_cast<uint32_t *>(c);
    MmFold &f = *fp;
    int rc = fold_matmul(x, y, &f);
    if (rc) return rc;
    const int64_t M = f.M, N = f.N, K = f.K, batch = f.batch;
    const int w = f.nb;
    a.a_sm = f.a_sm;
    a.a_sk = f.a_sk;
    a.b_sk = f.b_sk;
    a.b_sn = f.b_sn;
    if (M > 0x7FFFFFFFll || N > 0x7FFFFFFFll || K > 0x7FFFFFFFll || batch > 65535ll * 1024)
        return fail(CG_ERR_UNSUPPORTED, "matmul: extent above 2^31-1");
    a.M = (uint32_t)M;
    a.N = (uint32_t)N;
    a.K = (uint32_t)K;
    a.nb = (uint32_t)w;
    a.batch = (uint32_t)batch;
    for (int d = 0; d < w; d++) {
        a.bd[d] = (uint32_t)f.bd[d];
        a.bdiv[d] = make_fastdiv(a.bd[d]);
        a.a_bs[d] = f.a_bs[d];
        a.b_bs[d] = f.b_bs[d];
    }
    return CG_OK;
}

// The 32-bit words of one operand (`left`: x, else y) and whether 16-byte loads may run along its unit-stride axis.  An
// operand that lies in memory in a narrow format is read through its widened copy, unless the caller takes it as it
// lies (`native`: then the address stays null and the operand counts as unaligned).
static int mm_operand(const cg_tensor *t, bool left, bool native, MmArgs *ap) {
    MmArgs &a = *ap;
    const void *p = nullptr;
    if (!native) {
        int rc = device_ptr(t, &p);
        if (rc) return rc;
    }
    bool al = !native && reinterpret_cast<uintptr_t>(p) % 16 == 0;
    for (uint32_t d = 0; d < a.nb; d++)
        if ((left ? a.a_bs[d] : a.b_bs[d]) % 4) al = false;
    // 16-byte loads run along the unit-stride axis; the other axis' stride must keep alignment
    if (left) {
        a.A = static_cast<const uint32_t *>(p);
        const bool kfast = a.a_sk == 1 || a.K == 1, mfast = !kfast && a.a_sm == 1;
        a.a_vec = al && ((a.a_sk == 1 && a.a_sm % 4 == 0) || (mfast && a.a_sk % 4 == 0));
    } else {
        a.B = static_cast<const uint32_t *>(p);
        const bool kfast = a.b_sk == 1 || a.K == 1, nfast = !kfast && a.b_sn == 1;
        a.b_vec = al && ((a.b_sk == 1 && a.b_sn % 4 == 0) || (nfast && a.b_sk % 4 == 0));
    }
    return CG_OK;
}

static int make_mm_args(const cg_tensor *x, const cg_tensor *y, void *c, MmArgs *ap, MmFold *fp) {
    int rc = mm_geometry(x, y, c, ap, fp);
    if (!rc) rc = mm_operand(x, true, false, ap);
    if (!rc) rc = mm_operand(y, false, false, ap);
    return rc;
}

// The buffer that device_ptr's address of t lies in: the widened copy for a view of a narrow buffer.
static Buffer *words_buffer(const cg_tensor *t) { return is_narrow_buf(t->buf) ? t->buf->wide : t->buf; }

// May the [rows, K] view of t (row stride s_r, k stride s_k, in elements) be multiplied as it lies in memory, by the
// kernels of narrow kind `kind` (1 bf16, 2 f16, 3 fp8)?  Its buffer holds that very format, k is contiguous and every row
// starts on a 16-byte boundary.  dense: the rows must also follow each other without gaps.
static bool native_rows(const cg_tensor *t, int kind, int64_t s_r, int64_t s_k, int64_t K, bool dense) {
    if (!t->buf || t->uniform || t->buf->fmt != kind) return false;
    const int64_t eb = (int64_t)fmt_bytes(kind);
    if (s_k != 1 || s_r * eb % 16 != 0 || t->offset * eb % 16 != 0) return false;
    return !dense || s_r == K;
}
static const void *native_ptr(const cg_tensor *t) {
    return static_cast<const char *>(t->buf->ptr) + t->offset * (int64_t)fmt_bytes(t->buf->fmt);
}

// One to eight rows, k contiguous in 16-byte pieces, one batch entry: skinny.hpp
static SkinnyInput skinny_input(const MmArgs &a, const NormFuse *nf) {
    SkinnyInput in = {reinterpret_cast<const float *>(a.A), nullptr, a.a_sm, a.M, a.K, 0, 0, 0};
    if (nf) {
        in.gamma = reinterpret_cast<const float *>(nf->gamma);
        in.n_bits = nf->n_bits;
        in.eps_bits = nf->eps_bits;
        in.exp_bits = nf->exp_bits;
    }
    return in;
}
static SkinnyProduct skinny_product(const MmArgs &a) { // its rows stored as they are
    return {reinterpret_cast<const float *>(a.B), a.b_sn, a.N, 0, a.C, a.N, 0, nullptr, nullptr, a.N, 0};
}
// Whether a product that shares its launch with no other goes there too: where enough of the lanes' loads are values, `least` sixteenths of a
// whole cut of k (see with_cut).  What is enough differs by the rows that share a lane's weights, by the columns (from 8192 on eight a
// workgroup) and, from 16384 columns on, where the other side is skinny_kt_wide_kernel.  Weights from memory, us a launch on the other side and here:
//   1 row    4096 x 8190 26.1, 22.9; 2304 x 4096 10.4, 8.7; 576 x 4096 5.1, 4.8; less than 9 / 16: 1028 x 12288 11.5, 12.6; 260 x 8190 5.0, 5.6
//   2 rows   3584 x 8190 23.4, 20.5; 2052 x 4096 9.2, 9.2; 260 x 16384 9.9, 7.6; but 1028 x 4096 6.1, 6.9
//   4 rows   3584 x 4096 14.6, 13.8; 4100 x 12288 40.0, 36.4; 2880 x 32768 70.2, 66.9; 260 x 16384 10.4, 9.6; but 2560 x 8190 19.2, 21.8; 2304 x 16384 29.7, 31.9
//   8 rows   3584 x 3584 29.6, 17.4; 2304 x 8190 32.1, 27.2; 5120 x 8194 60.8, 46.8; 960 x 32768 34.2, 26.9; but 2052 x 12288 36.1, 41.5; 3072 x 16384 49.2, 58.6
static bool skinny_alone(const MmArgs &a) {
    const uint32_t M = a.M, K = a.K, cut = M > 1 ? (K <= 1024 ? 1024 : 2048) : K <= 4096 ? 1024 : K <= 6144 ? 6144 : 8192, whole = (K + cut - 1) / cut * cut;
    const bool many = a.N >= 16384, rounds = M > 1 && K > 2048;
    uint32_t least = 9;
    if (M > 1 && K > 6144) least = 0; // (one idle part of four rounds and more: 8 x 9216 x 18000 160.9, 135)
    else if (M == 2) least = many || rounds ? 0 : 9;
    else if (M > 2 && M <= 4) least = rounds ? (K > 4096 ? 0 : many ? 11 : 14) : many && K <= 1024 ? 0 : 9;
    else if (M > 4 && many) least = K <= 1024 ? 12 : 15;
    else if (M > 4 && rounds && a.N >= 8192) least = M > 6 ? 9 : 13; // (this side takes as long for five rows as for eight: 2560 x 12288 37.5 and 42.0, 46.1 and 42.8)
    return 16ull * K >= (uint64_t)least * whole;
}
static bool skinny_operands(const MmArgs &a) { return a.a_vec && a.b_vec && a.a_sk == 1 && a.b_sk == 1 && takes_skinny(a.M, a.K); }

int launch_matmul_group(cg_backend *be, const cg_tensor *x, const cg_tensor *const *ys, cg_tensor *const *outs, int n,
                        const NormFuse *nf) {
    if (int frc = flush_deferred(be)) return frc;
    if (n < (nf ? 1 : 2) || n > kMaxSkinny || x->dt != CG_F32) return kDeclined;
    SkinnyGroup g = {};
    MmArgs first;
    double bytes = distinct_bytes(x);
    for (int i = 0; i < n; i++) {
        MmArgs a;
        MmFold f;
        int rc = make_mm_args(x, ys[i], outs[i]->buf->ptr, &a, &f);
        if (rc) return rc;
        if (f.batch != 1 || !skinny_operands(a) || a.N < 4) return kDeclined;
        if (i == 0) first = a;
        else if (a.M != first.M || a.K != first.K || a.a_sm != first.a_sm) return kDeclined;
        g.p[i] = skinny_product(a);
        bytes += distinct_bytes(ys[i]) + distinct_bytes(outs[i]);
    }
    g.in = skinny_input(first, nf);
    g.count = (uint32_t)n;
    ProfScope prof(be, CG_K_GEMM_SKINNY, bytes);
    return launch_skinny_group(be, g);
}

int launch_matmul_group_rope(cg_backend *be, const cg_tensor *x, const cg_tensor *const *ys, const RopeStore *stores, int n,
                             const NormFuse *nf) {
    if (n < 1 || n > kMaxSkinny || x->dt != CG_F32) return kDeclined;
    SkinnyGroup g = {};
    MmArgs first;
    double bytes = distinct_bytes(x);
    bool by_head = false; // some product's heads are normed: two launches (see head_norm_rope_finish_kernel)
    for (int i = 0; i < n; i++) by_head = by_head || stores[i].hgamma != nullptr;
    for (int i = 0; i < n; i++) {
        MmArgs a;
        MmFold f;
        int rc = make_mm_args(x, ys[i], stores[i].dst, &a, &f);
        if (rc) return rc;
        const RopeStore &st = stores[i];
        if (f.batch != 1 || !skinny_operands(a) || a.N >= 8192) return kDeclined;
        if (i == 0) first = a;
        else if (a.M != first.M || a.K != first.K || a.a_sm != first.a_sm) return kDeclined;
        if (st.hd < 8 || st.hd % 8 || a.N % st.hd || !st.dst || (st.rope && (!st.cos || !st.sin))) return kDeclined;
        if (by_head && (st.hd % 16 || st.hd > 128)) return kDeclined;
        g.p[i] = {reinterpret_cast<const float *>(a.B), a.b_sn, a.N, 0, st.dst, st.sb, st.sh, st.cos, st.sin, st.hd, st.rope};
        bytes += distinct_bytes(ys[i]) + 4.0 * (double)a.M * a.N;
    }
    g.in = skinny_input(first, nf);
    g.count = (uint32_t)n;
    ProfScope prof(be, CG_K_GEMM_SKINNY, bytes);
    if (!by_head) return launch_skinny_group(be, g);
    uint64_t words = 0; // the normed products go to scratch memory as they are
    for (int i = 0; i < n; i++)
        if (stores[i].hgamma) words += (uint64_t)first.M * g.p[i].n;
    void *scratch = nullptr;
    size_t cls = 0;
    if (int arc = be->pool.alloc(words * 4, &scratch, &cls)) return arc;
    OpenHeads *const heads = new OpenHeads;
    heads->rows = first.M;
    heads->scratch = scratch;
    heads->cls = cls;
    uint32_t *at = static_cast<uint32_t *>(scratch);
    for (int i = 0; i < n; i++) {
        if (!stores[i].hgamma) continue;
        SkinnyProduct &p = g.p[i]; // column n of row m to at[m * N + n]
        heads->p[heads->count++] = {stores[i], at, p.n};
        p.dst = at;
        p.sb = p.n;
        p.sh = stores[i].hd;
        p.rope = 0;
        at += (uint64_t)first.M * p.n;
    }
    be->heads = heads;
    const int rc = launch_skinny_group(be, g);
    if (rc) drop_open_heads(be);
    return rc;
}

void drop_open_heads(cg_backend *be) {
    OpenHeads *const h = be->heads;
    be->heads = nullptr;
    be->pool.free(h->scratch, h->cls); // stream-ordered: later users queue behind the launch that reads it
    for (Buffer *b : h->held) buffer_release(b);
    delete h;
}

int launch_open_heads(cg_backend *be) {
    const OpenHeads &h = *be->heads;
    HeadFinish f;
    memset(&f, 0, sizeof f);
    f.n = h.count;
    f.M = h.rows;
    uint32_t heads = 0, hd = 0;
    for (uint32_t i = 0; i < h.count; i++) {
        f.s[i] = h.p[i].to;
        f.src[i] = h.p[i].src;
        f.N[i] = h.p[i].n;
        heads = std::max(heads, h.p[i].n / h.p[i].to.hd);
        hd = std::max(hd, h.p[i].to.hd);
    }
    ProfScope prof(be, CG_K_GEMM_SKINNY, 8.0 * f.M * heads * hd * f.n);
    launch_kernel(head_norm_rope_finish_kernel, dim3(heads, f.n), dim3((f.M * hd + 63) / 64 * 64), 0, be->stream, f);
    const hipError_t e = hipGetLastError();
    drop_open_heads(be);
    return e == hipSuccess ? CG_OK : hip_fail(e, "head norm launch");
}

// out = g * (1 / (one + exp(-g))) * u with g = x.yg, u = x.yu: two decode-time linear layers and
// the program between them and the next product in one launch.
int launch_matmul_gated(cg_backend *be, const cg_tensor *x, const cg_tensor *yg, const cg_tensor *yu, uint32_t one,
                        cg_tensor *out, const NormFuse *nf) {
    if (int frc = flush_deferred(be)) return frc;
    if (x->dt != CG_F32) return kDeclined;
    MmArgs ag, au;
    MmFold fg, fu;
    uint32_t *const c = static_cast<uint32_t *>(out->buf->ptr) + out->offset; // out: a contiguous view, not always at element 0
    int rc = make_mm_args(x, yg, c, &ag, &fg);
    if (!rc) rc = make_mm_args(x, yu, c, &au, &fu);
    if (rc) return rc;
    if (fg.batch != 1 || fu.batch != 1 || !skinny_operands(ag) || !skinny_operands(au) || ag.N < 512 || au.N != ag.N || au.K != ag.K || au.M != ag.M || au.b_sn != ag.b_sn)
        return kDeclined;
    if (ag.M > 4 && !nf) return kDeclined; // (more than four rows: a decode step's, whose norm comes along; others as a grouped product and the program)
    ProfScope prof(be, CG_K_GEMM_SKINNY, distinct_bytes(x) + distinct_bytes(yg) + distinct_bytes(yu) + distinct_bytes(out));
    return launch_skinny_gated(be, {skinny_input(ag, nf), reinterpret_cast<const float *>(ag.B), reinterpret_cast<const float *>(au.B), ag.b_sn, ag.N, one, c});
}

// out = a sum of two or four terms, term[slot] = x.y, the others dense tensors of out's shape (device pointers); `order` as in SkinnyResidual.
int launch_matmul_residual(cg_backend *be, const cg_tensor *x, const cg_tensor *y, const uint32_t *const *terms, int nterms,
                           int slot, int order, cg_tensor *out) {
    if (int frc = flush_deferred(be)) return frc;
    if (x->dt != CG_F32) return kDeclined;
    MmArgs a;
    MmFold f;
    int rc = make_mm_args(x, y, static_cast<uint32_t *>(out->buf->ptr) + out->offset, &a, &f);
    if (rc) return rc;
    if (f.batch != 1 || !skinny_operands(a) || a.N < 512 || a.N >= 8192) return kDeclined;
    SkinnyResidual r = {skinny_input(a, nullptr), reinterpret_cast<const float *>(a.B), a.b_sn, a.N, {}, (uint32_t)slot, (uint32_t)order, (uint32_t)nterms, a.C};
    for (int t = 0; t < nterms; t++) r.term[t] = t == slot ? nullptr : terms[t];
    ProfScope prof(be, CG_K_GEMM_SKINNY, distinct_bytes(x) + distinct_bytes(y) + 4.0 * distinct_bytes(out));
    return launch_skinny_residual(be, r);
}

// ---- narrow operands for the 16-bit and 8-bit matrix instructions ---------------------------------------------------
// A [rows, k] view of f32 words that hold values of a narrow dtype (exactly) is written as its 2-byte (bf16 / f16) or
// 1-byte (fp8) patterns, k contiguous: half or a quarter of the bytes for the product that follows, and a tile of the
// same 32 words is 64 or 128 deep in k.  KIND 1 bf16, 2 f16, 3 fp8.  A thread narrows four consecutive k of a row.
template <int KIND>
__global__ __launch_bounds__(kThreads) void pack_operand_kernel(const uint32_t *src, int64_t s_r, int64_t s_k, uint32_t rows, uint32_t K,
                                                                void *dst) {
    const uint64_t quads = (uint64_t)rows * (K / 4);
    const uint64_t i = (uint64_t)blockIdx.x * kThreads + threadIdx.x;
    if (i >= quads) return;
    const uint32_t r = (uint32_t)(i / (K / 4)), k = (uint32_t)(i % (K / 4)) * 4;
    const uint32_t *p = src + (int64_t)r * s_r + (int64_t)k * s_k;
    uint32_t w[4];
    if (s_k == 1 && ((reinterpret_cast<uintptr_t>(p) & 15) == 0)) {
        const uint4 v = *reinterpret_cast<const uint4 *>(p);
        w[0] = v.x, w[1] = v.y, w[2] = v.z, w[3] = v.w;
    } else {
#pragma unroll
        for (int e = 0; e < 4; e++) w[e] = p[(int64_t)e * s_k];
    }
    if constexpr (KIND == 3) {
        static_cast<uint32_t *>(dst)[i] = (uint32_t)f8_byte_of(w[0]) | ((uint32_t)f8_byte_of(w[1]) << 8) | ((uint32_t)f8_byte_of(w[2]) << 16) |
                                          ((uint32_t)f8_byte_of(w[3]) << 24);
    } else {
        uint2 o;
        o.x = pack_halves<KIND>(asf(w[0]), asf(w[1]));
        o.y = pack_halves<KIND>(asf(w[2]), asf(w[3]));
        static_cast<uint2 *>(dst)[i] = o;
    }
}

// (env CG_GEMM_PACKED=0 keeps the products of narrow dtypes on 32-bit words)
static bool packed_narrow_ok() {
    static const bool ok = [] {
        const char *e = getenv("CG_GEMM_PACKED");
        return !(e && e[0] == '0');
    }();
    return ok;
}

// (env CG_PACKED_MFMA=0 keeps few-row products of the 16-bit dtypes on the wave-per-column kernel, for measurements)
static bool packed_mfma_ok() {
    static const bool ok = [] {
        const char *e = getenv("CG_PACKED_MFMA");
        return !(e && e[0] == '0');
    }();
    return ok;
}

// The narrow copy of the [rows, K] view (row stride s_r, k stride s_k, in words) at `ptr` inside `buf`: the copy kept with
// the buffer for this very view if there is one; else a new one, kept with the buffer when `keep` (a weight matrix is
// narrowed once, shared activations once for the products that multiply them; the oldest entry makes room when the list is
// full), else handed to the caller, who frees *tmp after its launch.
static int pack_operand(cg_backend *be, Buffer *buf, const uint32_t *ptr, int64_t s_r, int64_t s_k, int64_t rows, int64_t K, int kind,
                        bool keep, const void **packed, void **tmp, size_t *tmp_cls) {
    const int64_t off = ptr - static_cast<const uint32_t *>(buf->ptr);
    for (const Buffer::Packed &p : buf->packed)
        if (p.kind == kind && p.off == off && p.rows == rows && p.k == K && p.sr == s_r && p.sk == s_k) {
            *packed = p.ptr;
            return CG_OK;
        }
    void *dst = nullptr;
    size_t cls = 0;
    int rc = be->pool.alloc((size_t)rows * (size_t)K * (kind == 3 ? 1 : 2), &dst, &cls);
    if (rc) return rc;
    const uint64_t quads = (uint64_t)rows * (uint64_t)(K / 4);
    const dim3 grid((uint32_t)((quads + kThreads - 1) / kThreads));
    {
        ProfScope prof(be, CG_K_PACK, (double)rows * (double)K * (4.0 + (kind == 3 ? 1.0 : 2.0)));
        if (kind == 1) launch_kernel(pack_operand_kernel<1>, grid, dim3(kThreads), 0, be->stream, ptr, s_r, s_k, (uint32_t)rows, (uint32_t)K, dst);
        else if (kind == 2) launch_kernel(pack_operand_kernel<2>, grid, dim3(kThreads), 0, be->stream, ptr, s_r, s_k, (uint32_t)rows, (uint32_t)K, dst);
        else launch_kernel(pack_operand_kernel<3>, grid, dim3(kThreads), 0, be->stream, ptr, s_r, s_k, (uint32_t)rows, (uint32_t)K, dst);
    }
    if (keep) {
        if (buf->packed.size() >= kMaxPackedPerBuffer) { // stream-ordered free: products already queued on it come first
            be->pool.free(buf->packed.front().ptr, buf->packed.front().cls);
            buf->packed.erase(buf->packed.begin());
        }
        Buffer::Packed p;
        p.ptr = dst;
        p.cls = cls;
        p.kind = kind;
        p.off = off;
        p.rows = rows;
        p.k = K;
        p.sr = s_r;
        p.sk = s_k;
        buf->packed.push_back(p);
    } else {
        *tmp = dst;
        *tmp_cls = cls;
    }
    *packed = dst;
    return CG_OK;
}

// Few rows (M <= 8) times a weight matrix of a narrow dtype that pack_operand narrowed in memory: a wave per output
// column walks K with 16-byte loads of the narrow row (8 two-byte or 16 one-byte weights per lane and trip), widens them in
// registers (exact) and multiplies with the f32 words of the activations; HBM-bound on the narrow weights, 2 or 1 bytes
// per weight instead of 4.  f32 accumulation, lanes combined by a wave shuffle.  KIND 1 bf16, 2 f16, 3 fp8.
template <int KIND> __device__ __forceinline__ void widen_weights(const uint4v &raw, float (&w)[KIND == 3 ? 16 : 8]) {
    const uint32_t r[4] = {raw[0], raw[1], raw[2], raw[3]};
    if constexpr (KIND == 1) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            w[2 * i] = asf(r[i] << 16);
            w[2 * i + 1] = asf(r[i] & 0xFFFF0000u);
        }
    } else if constexpr (KIND == 2) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            w[2 * i] = __half2float(__ushort_as_half((unsigned short)(r[i] & 0xFFFFu)));
            w[2 * i + 1] = __half2float(__ushort_as_half((unsigned short)(r[i] >> 16)));
        }
    } else {
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int b = 0; b < 4; b++) w[4 * i + b] = asf(f8_word_of((uint8_t)(r[i] >> (8 * b))));
    }
}
// The same for at most four rows of the 16-bit dtypes on the matrix instruction v_mfma_f32_4x4x4_{bf16_1k,f16}: the layout
// of skinny_kt_mfma_xreg_kernel (lane (b, j) = (lane / 4, lane % 4) feeds weight row n0 + j and activation row j for the k of
// block b) with 8 k per lane and trip instead of 4: one 16-byte load of narrow weights drives two instructions.  The
// activations, which are f32 words in memory, are narrowed (exact) into registers ONCE per workgroup — all of K, 16
// registers per 2048 — and the workgroup walks `iters` consecutive groups of four columns with them, the next group's
// weights on their way while the current group is reduced: the activation traffic out of L2, twice the weights' bytes per
// column group, is paid once.  K = KCH x 1024.  KIND 1 bf16, 2 f16.
typedef short short4v __attribute__((ext_vector_type(4)));
typedef _Float16 half4v __attribute__((ext_vector_type(4)));
template <int KIND, int KCH>
__global__ __launch_bounds__(kThreads) void skinny_kt_packed_mfma_kernel(const MmArgs a, const void *weights, uint32_t iters) {
    constexpr int TRIPS = 2 * KCH; // a wave takes 128 k per trip, four waves 512: two trips per 1024
    const uint32_t wave = threadIdx.x / 64, lane = threadIdx.x % 64;
    const uint32_t j = lane % 4, b = lane / 4;
    const uint32_t kb = wave * 128 + b * 8; // this lane's k: kb + 512 t .. + 7
    const uint32_t groups = (a.N + 3) / 4;
    const uint32_t first_grp = blockIdx.x * iters;
    if (first_grp >= groups) return; // the same for every thread of the workgroup
    uint4v wq[TRIPS];
    auto ask = [&](uint32_t grp) {
        const uint16_t *row = static_cast<const uint16_t *>(weights) + (size_t)min(grp * 4 + j, a.N - 1) * a.K + kb;
#pragma unroll
        for (int t = 0; t < TRIPS; t++) wq[t] = __builtin_nontemporal_load(reinterpret_cast<const uint4v *>(row + 512 * t));
    };
    ask(first_grp);
    // the activations of row j, narrowed: xq[t] = its 8 values at kb + 512 t as four words of two
    uint4v xq[TRIPS];
    {
        const uint32_t *xrow = a.A + (int64_t)min(j, a.M - 1) * a.a_sm + kb;
#pragma unroll
        for (int t = 0; t < TRIPS; t++) {
            const float4v lo = *reinterpret_cast<const float4v *>(xrow + 512 * t), hi = *reinterpret_cast<const float4v *>(xrow + 512 * t + 4);
            xq[t][0] = pack_halves<KIND>(lo[0], lo[1]);
            xq[t][1] = pack_halves<KIND>(lo[2], lo[3]);
            xq[t][2] = pack_halves<KIND>(hi[0], hi[1]);
            xq[t][3] = pack_halves<KIND>(hi[2], hi[3]);
        }
    }
    __shared__ float part[2][4][16];
    for (uint32_t it = 0; it < iters; it++) {
        const uint32_t grp = first_grp + it;
        if (grp >= groups) break;
        float4v acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < TRIPS; t++) {
            typedef uint32_t uint2v __attribute__((ext_vector_type(2)));
            const uint2v x0 = {xq[t][0], xq[t][1]}, x1 = {xq[t][2], xq[t][3]}, w0 = {wq[t][0], wq[t][1]}, w1 = {wq[t][2], wq[t][3]};
            if constexpr (KIND == 1) {
                acc = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(__builtin_bit_cast(short4v, x0), __builtin_bit_cast(short4v, w0), acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(__builtin_bit_cast(short4v, x1), __builtin_bit_cast(short4v, w1), acc, 0, 0, 0);
            } else {
                acc = __builtin_amdgcn_mfma_f32_4x4x4f16(__builtin_bit_cast(half4v, x0), __builtin_bit_cast(half4v, w0), acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_f32_4x4x4f16(__builtin_bit_cast(half4v, x1), __builtin_bit_cast(half4v, w1), acc, 0, 0, 0);
            }
        }
        if (it + 1 < iters && grp + 1 < groups) ask(grp + 1); // on its way through the reduction of this group
        float (*pt)[16] = part[it & 1];
        const float v = four_sums(acc[0], acc[1], acc[2], acc[3]);
        if (lane / 4 % 4 == 0) pt[wave][lane / 4 + j] = v;
        __syncthreads(); // (the buffer written two groups ago was read before the barrier of the group in between)
        if (threadIdx.x < 16) {
            const uint32_t m = threadIdx.x / 4, col = grp * 4 + threadIdx.x % 4;
            const float v = (pt[0][threadIdx.x] + pt[1][threadIdx.x]) + (pt[2][threadIdx.x] + pt[3][threadIdx.x]);
            if (col < a.N && m < a.M) a.C[(uint64_t)m * a.N + col] = asu(v);
        }
    }
}

template <int MM, int KIND>
__global__ __launch_bounds__(kThreads) void skinny_kt_packed_kernel(const MmArgs a, const void *weights) {
    constexpr int PER = KIND == 3 ? 16 : 8; // weights per lane and trip
    const uint32_t wave = threadIdx.x / 64, lane = threadIdx.x % 64;
    const uint32_t n = blockIdx.x * 4 + wave;
    if (n >= a.N) return;
    const uint8_t *row = static_cast<const uint8_t *>(weights) + (size_t)n * a.K * (KIND == 3 ? 1 : 2);
    float acc[MM];
#pragma unroll
    for (int m = 0; m < MM; m++) acc[m] = 0.0f;
#pragma unroll 2
    for (uint32_t k = lane * PER; k < a.K; k += 64 * PER) {
        const uint4v raw = __builtin_nontemporal_load(reinterpret_cast<const uint4v *>(row + (size_t)k * (KIND == 3 ? 1 : 2)));
        float w[PER];
        widen_weights<KIND>(raw, w);
#pragma unroll
        for (int m = 0; m < MM; m++) {
            if ((uint32_t)m < a.M) {
                const uint32_t *x = a.A + (int64_t)m * a.a_sm + k;
#pragma unroll
                for (int q = 0; q < PER / 4; q++) {
                    const float4v xv = *reinterpret_cast<const float4v *>(x + 4 * q);
                    acc[m] = fmaf(xv[0], w[4 * q], acc[m]);
                    acc[m] = fmaf(xv[1], w[4 * q + 1], acc[m]);
                    acc[m] = fmaf(xv[2], w[4 * q + 2], acc[m]);
                    acc[m] = fmaf(xv[3], w[4 * q + 3], acc[m]);
                }
            }
        }
    }
#pragma unroll
    for (int m = 0; m < MM; m++) {
        acc[m] = wave_add<1>(acc[m]);
        if (lane == 0 && (uint32_t)m < a.M) a.C[(uint64_t)m * a.N + n] = asu(acc[m]);
    }
}

// x . y -> out on the 128-wide tiles, an operand that does not lie narrow packed first.  kDeclined: the pool has no room for that.
static int low_product(cg_backend *be, int kind, const cg_tensor *x, bool x_lies, const cg_tensor *y, bool y_lies, MmArgs a, int64_t M, int64_t N, int64_t K,
                       cg_tensor *out) {
    int rc = mm_operand(x, true, x_lies, &a);
    if (!rc) rc = mm_operand(y, false, y_lies, &a);
    if (rc) return rc;
    const void *pa = x_lies ? native_ptr(x) : nullptr, *pb = y_lies ? native_ptr(y) : nullptr;
    void *ta = nullptr, *tb = nullptr;
    size_t ca = 0, cb = 0;
    rc = x_lies ? CG_OK : pack_operand(be, words_buffer(x), a.A, a.a_sm, a.a_sk, M, K, kind, x->rc.load() > 1 || x->buf->rc.load() > 1, &pa, &ta, &ca);
    if (!rc && !y_lies) rc = pack_operand(be, words_buffer(y), a.B, a.b_sn, a.b_sk, N, K, kind, true, &pb, &tb, &cb);
    if (rc) {
        (void)hipGetLastError();
        rc = kDeclined;
    } else {
        ProfScope prof(be, CG_K_GEMM_MFMA, 2.0 * (double)M * (double)N * (double)K);
        rc = launch_narrow_tiles(be, kind, pa, x_lies ? a.a_sm : K, M, pb, y_lies ? a.b_sn : K, N, K, out->buf->ptr, out->buf->fmt);
    }
    if (ta) be->pool.free(ta, ca); // stream-ordered: later users queue behind the product
    if (tb) be->pool.free(tb, cb);
    return rc;
}

// patterns: operands of a narrow dtype may be multiplied from patterns; kDeclined: they would be, and the pool has no room to pack one.
static int product(cg_backend *be, const cg_tensor *x, const cg_tensor *y, cg_tensor *out, bool wide_only, bool patterns) {
    if (int frc = flush_deferred(be)) return frc;
    MmArgs a;
    MmFold f;
    int rc = mm_geometry(x, y, out ? out->buf->ptr : nullptr, &a, &f);
    if (rc) return rc;
    const int64_t M = f.M, N = f.N, K = f.K, batch = f.batch;
    const bool a_mfast = !(a.a_sk == 1 || K == 1) && a.a_sm == 1;
    const bool b_nfast = !(a.b_sk == 1 || K == 1) && a.b_sn == 1;

    if (batch > 65535) return fail(CG_ERR_UNSUPPORTED, "matmul: more than 65535 batch entries after folding");
    const bool f32 = is_f(x->dt);
    const int half = x->dt == CG_BF16 ? 1 : x->dt == CG_F16 ? 2 : 0; // operands of the 16-bit matrix instructions
    const int kind = half ? half : x->dt == CG_F8 ? 3 : 0;           // the narrow kernels' operand format (0: none)
    LaunchQueue &s = be->stream;

    // ---- the narrow dtypes' tiled kernels' plan (used by the last branch below; here because it decides how operands are addressed) ----
    // the 256 x 256 tile when it covers half of the chip (1024 x 2048 x 8192, 128 tiles: 53 us against 57 on 128 x 128 tiles, bf16;
    // 2048 x 2048 x 2048, 64 tiles: 46 against 39), all of it for fp8, whose instructions keep less of a sum (env CG_GEMM_BIG=0 switches it off)
    const uint64_t tiles_big = (uint64_t)((M + 255) / 256) * ((N + 255) / 256) * batch;
    static const bool big_allowed = [] {
        const char *e = getenv("CG_GEMM_BIG");
        return !(e && e[0] == '0');
    }();
    const bool big = big_allowed && kind && tiles_big >= (kind == 3 ? 256 : 128) && M >= 256 && N >= 256;
    // Operands of a narrow dtype are multiplied from 2-byte / 1-byte patterns where rows of k are whole 16-byte pieces: as they
    // lie in memory when their buffer holds that format, else narrowed in memory first (the right operand once per buffer)
    // (env CG_GEMM_PACKED=0 switches it off).
    const bool packable = patterns && f32 && K != 0 && M > 8 && kind && packed_narrow_ok() && batch == 1 && K % (kind == 3 ? 16 : 8) == 0 && x->buf && y->buf;
    const bool x_lies = packable && native_rows(x, kind, a.a_sm, a.a_sk, K, false), y_lies = packable && native_rows(y, kind, a.b_sn, a.b_sk, K, false);
    const NarrowRoute route = narrow_route(kind, {M, a.a_sm, x_lies}, {N, a.b_sn, y_lies}, K, packable, big, wide_only);
    const bool big_packed = route == NarrowRoute::wide, low = route == NarrowRoute::low;
    const bool x_native = (big_packed || low) && x_lies, y_native_rows = (big_packed || low) && y_lies;
    // Whole stages of 64 bytes of k in whole turns of the ring, 16-byte rows, byte offsets that fit 32 bits: the wide tile
    // fed by loads straight into LDS (env CG_GEMM_DLDS=0: the register-staged one).  Only that kernel can round the result
    // to the operands' format in its store; without `out` the call just says whether this product would run on it.
    static const bool dlds_allowed = [] {
        const char *e = getenv("CG_GEMM_DLDS");
        return !(e && e[0] == '0');
    }();
    const int64_t per = kind == 3 ? 4 : 2;           // elements per 32-bit word
    const int64_t kw = kind ? K / per : 0;           // words per row
    const int64_t a_pitch = x_native ? a.a_sm / per : kw, b_pitch = y_native_rows ? a.b_sn / per : kw; // (a view taken as it lies keeps its own row pitch)
    const bool dlds = big_packed && dlds_allowed && kw % (16 * kDldsStages) == 0 && a_pitch % 4 == 0 && b_pitch % 4 == 0 &&
                      (!x_native || reinterpret_cast<uintptr_t>(native_ptr(x)) % 16 == 0) && (!y_native_rows || reinterpret_cast<uintptr_t>(native_ptr(y)) % 16 == 0) &&
                      (uint64_t)M * (uint64_t)a_pitch * 4 < (1ull << 32) && (uint64_t)N * (uint64_t)b_pitch * 4 < (1ull << 32) &&
                      (uint64_t)M * (uint64_t)N < (1ull << 30);
    const bool can_round = (dlds && N % 4 == 0) || low;
    if (!out) return can_round ? CG_OK : kDeclined;

    // ---- the operands' addresses -------------------------------------------------------------------------------------
    if (low) return low_product(be, kind, x, x_native, y, y_native_rows, a, M, N, K, out);
    rc = mm_operand(x, true, x_native, &a);
    if (rc) return rc;
    // a decode-time linear layer of a narrow dtype reads its weight matrix at 2 or 1 bytes a weight (see below)
    const bool skinny_packed = f32 && K != 0 && M <= (half ? 8 : 2) && packed_narrow_ok() && kind && batch == 1 && a.a_sk == 1 && a.a_vec &&
                               a.a_sm % 4 == 0 && K % 16 == 0 && K >= 256 && N >= 64 && y->buf;
    const bool y_native = (skinny_packed && native_rows(y, kind, a.b_sn, a.b_sk, K, true)) || y_native_rows;
    rc = mm_operand(y, false, y_native, &a);
    if (rc) return rc;
    const int c_fmt = out->buf->fmt;
    if (c_fmt != kFmtWords && !can_round) return fail(CG_ERR_ARG, "matmul: a narrow result needs the kernel that rounds in its store");
    const double flop = 2.0 * (double)M * (double)N * (double)K * (double)batch;
    const double bytes = distinct_bytes(x) + distinct_bytes(y) + distinct_bytes(out);
    const bool simple = K == 0 || !f32, skinny = !simple && M <= 8 && (a.b_sk == 1 || a.b_sn == 1);
    ProfScope prof(be, simple ? CG_K_GEMM_SIMPLE : skinny ? CG_K_GEMM_SKINNY : CG_K_GEMM_MFMA, skinny ? bytes : flop);
    if (!simple && !skinny && !kind) return launch_split_gemm(be, a, a_mfast, b_nfast); // (no narrow dtype)
    if (K == 0 || !f32) {
        uint64_t elems = (uint64_t)M * N;
        dim3 grid((uint32_t)((elems + kThreads - 1) / kThreads), (uint32_t)batch);
        if (f32)
            launch_kernel((simple_gemm_kernel<true>), grid, dim3(kThreads), 0, s, a);
        else
            launch_kernel((simple_gemm_kernel<false>), grid, dim3(kThreads), 0, s, a);
    } else if (skinny_packed) {
        // a decode-time linear layer of a narrow dtype: the weight matrix in memory as its dtype's patterns (as uploaded, or
        // narrowed once), read at 2 or 1 bytes a weight
        // (measured on 2048 x 8192: one row 10.7 instead of 15.6 us for the 16-bit dtypes, 13.2 instead of 15.4 for fp8; with
        // four rows the loads of the activations bound both kernels alike, and widening fp8 costs more than it saves)
        const void *pb = y_native ? native_ptr(y) : nullptr;
        void *tb = nullptr;
        size_t cb = 0;
        int prc = y_native ? CG_OK : pack_operand(be, words_buffer(y), a.B, a.b_sn, a.b_sk, N, K, kind, true, &pb, &tb, &cb);
        if (prc) return prc;
        const dim3 pgrid((uint32_t)((N + 3) / 4));
        const int kch = (int)(K / 1024);
        if (half && M <= 4 && K % 1024 == 0 && (kch == 1 || kch == 2 || kch == 4 || kch == 8) && packed_mfma_ok()) {
            // all of the activations narrowed into registers, several column groups per workgroup (see the kernel)
            const uint32_t groups = (uint32_t)((N + 3) / 4), iters = xreg_cols_iters(groups);
            const dim3 mgrid((groups + iters - 1) / iters);
#define CG_PACKED_MFMA(KCH)                                                                                              \
    if (half == 1) launch_kernel((skinny_kt_packed_mfma_kernel<1, KCH>), mgrid, dim3(kThreads), 0, s, a, pb, iters);      \
    else launch_kernel((skinny_kt_packed_mfma_kernel<2, KCH>), mgrid, dim3(kThreads), 0, s, a, pb, iters);
            if (kch == 1) { CG_PACKED_MFMA(1) }
            else if (kch == 2) { CG_PACKED_MFMA(2) }
            else if (kch == 4) { CG_PACKED_MFMA(4) }
            else { CG_PACKED_MFMA(8) }
#undef CG_PACKED_MFMA
            if (tb) be->pool.free(tb, cb);
            hipError_t me = hipGetLastError();
            return me == hipSuccess ? CG_OK : hip_fail(me, "matmul launch");
        }
#define CG_PACKED(MM)                                                                                                     \
    if (kind == 1) launch_kernel((skinny_kt_packed_kernel<MM, 1>), pgrid, dim3(kThreads), 0, s, a, pb);                  \
    else if (kind == 2) launch_kernel((skinny_kt_packed_kernel<MM, 2>), pgrid, dim3(kThreads), 0, s, a, pb);             \
    else launch_kernel((skinny_kt_packed_kernel<MM, 3>), pgrid, dim3(kThreads), 0, s, a, pb);
        if (M <= 1) { CG_PACKED(1) }
        else if (M <= 4) { CG_PACKED(4) }
        else { CG_PACKED(8) }
#undef CG_PACKED
        if (tb) be->pool.free(tb, cb); // stream-ordered: later users queue behind the product
    } else if (M <= 8 && a.b_sk == 1) {
        const bool vec = a.a_vec && a.b_vec && a.a_sk == 1 && K % 4 == 0;
#define CG_MM_SWITCH(CALL)        \
    if (M <= 1) { CALL(1) }       \
    else if (M <= 4) { CALL(4) }  \
    else { CALL(8) }
        if (!vec) {
            dim3 grid((uint32_t)((N + 3) / 4), (uint32_t)batch);
#define CG_CALL(MMV) launch_kernel((skinny_kt_kernel<MMV>), grid, dim3(kThreads), 0, s, a);
            CG_MM_SWITCH(CG_CALL)
#undef CG_CALL
        } else if (K <= 256) {
            const int lpc = K <= 64 ? 16 : K <= 128 ? 32 : 64;
            const uint32_t cols_per_block = 4 * (64 / lpc) * 4;
            dim3 grid((uint32_t)((N + cols_per_block - 1) / cols_per_block), (uint32_t)batch);
#define CG_CALL(MMV)                                                                                          \
    if (lpc == 16) launch_kernel((skinny_kt_narrow_kernel<MMV, 16>), grid, dim3(kThreads), 0, s, a);     \
    else if (lpc == 32) launch_kernel((skinny_kt_narrow_kernel<MMV, 32>), grid, dim3(kThreads), 0, s, a); \
    else launch_kernel((skinny_kt_narrow_kernel<MMV, 64>), grid, dim3(kThreads), 0, s, a);
            CG_MM_SWITCH(CG_CALL)
#undef CG_CALL
        } else {
            // enough waves to cover 256 CUs several times over, else split K inside the block
            const int64_t cols = N * batch;
            if (batch == 1 && cols >= 2048 && skinny_operands(a) && skinny_alone(a)) {
                const int orc = launch_skinny_group(be, {skinny_input(a, nullptr), {skinny_product(a)}, 1});
                if (orc) return orc;
            } else if (cols >= 16384) {
                dim3 grid((uint32_t)((N + 15) / 16), (uint32_t)batch);
#define CG_CALL(MMV) launch_kernel((skinny_kt_wide_kernel<MMV, 4, false>), grid, dim3(kThreads), 0, s, a);
                CG_MM_SWITCH(CG_CALL)
#undef CG_CALL
            } else if (cols >= 4096 && M <= 4) { // the wider projections of a decode step: activations are fetched once per 8 columns
                dim3 grid((uint32_t)((N + 7) / 8), (uint32_t)batch);
                xreg_either((uint32_t)K, xreg_trips((uint32_t)K), [&](auto whole) {
                    constexpr bool W = decltype(whole)::value;
                    if (xreg_trips((uint32_t)K) == 4)
                        launch_kernel((skinny_kt_mfma_xreg_kernel<W, 4, 2, 4>), grid, dim3(kThreads), 0, s, a);
                    else
                        launch_kernel((skinny_kt_mfma_xreg_kernel<W, 4, 2, 8>), grid, dim3(kThreads), 0, s, a);
                });
            } else if (cols >= 2048 && xreg_narrow((uint32_t)M, (uint32_t)K)) {
                dim3 grid((uint32_t)((N + 3) / 4), (uint32_t)batch);
                xreg_either((uint32_t)K, xreg_trips((uint32_t)K), [&](auto whole) {
                    constexpr bool W = decltype(whole)::value;
                    if (M > 4 && xreg_trips((uint32_t)K) == 4)
                        launch_kernel((skinny_kt_mfma_xreg_kernel<W, 8, 1, 4>), grid, dim3(kThreads), 0, s, a);
                    else if (M > 4)
                        launch_kernel((skinny_kt_mfma_xreg_kernel<W, 8, 1, 8>), grid, dim3(kThreads), 0, s, a);
                    else if (xreg_trips((uint32_t)K) == 4)
                        launch_kernel((skinny_kt_mfma_xreg_kernel<W, 4, 1, 4>), grid, dim3(kThreads), 0, s, a);
                    else
                        launch_kernel((skinny_kt_mfma_xreg_kernel<W, 4, 1, 8>), grid, dim3(kThreads), 0, s, a);
                });
            } else if (cols >= 2048) {
                dim3 grid((uint32_t)((N + 3) / 4), (uint32_t)batch);
#define CG_CALL(MMV) launch_kernel((skinny_kt_wide_kernel<MMV, 1, false>), grid, dim3(kThreads), 0, s, a);
                CG_MM_SWITCH(CG_CALL)
#undef CG_CALL
            } else {
                dim3 grid((uint32_t)N, (uint32_t)batch);
#define CG_CALL(MMV) launch_kernel((skinny_kt_wide_kernel<MMV, 1, true>), grid, dim3(kThreads), 0, s, a);
                CG_MM_SWITCH(CG_CALL)
#undef CG_CALL
            }
        }
    } else if (M <= 8 && a.b_sn == 1) {
        // split K over grid.z until about 2048 blocks are in flight (>= 128 k-rows each)
        const int64_t blocks_xy = ((N + 63) / 64) * batch;
        int64_t splits = std::min<int64_t>(std::min<int64_t>((2048 + blocks_xy - 1) / blocks_xy, (K + 127) / 128), 64);
        if (splits < 1) splits = 1;
        const uint32_t kchunk = (uint32_t)((((K + splits - 1) / splits) + 15) / 16 * 16);
        splits = (K + kchunk - 1) / kchunk;
        void *scratch = nullptr;
        size_t scratch_cls = 0;
        uint32_t *dst = a.C;
        if (splits > 1) {
            int prc = be->pool.alloc((size_t)batch * splits * M * N * 4, &scratch, &scratch_cls);
            if (prc) return prc;
            dst = static_cast<uint32_t *>(scratch);
        }
        dim3 grid((uint32_t)((N + 63) / 64), (uint32_t)batch, (uint32_t)splits);
#define CG_CALL(MMV) launch_kernel((skinny_nn_kernel<MMV>), grid, dim3(kThreads), 0, s, a, dst, kchunk);
        CG_MM_SWITCH(CG_CALL)
#undef CG_CALL
        if (splits > 1) {
            uint64_t total = (uint64_t)batch * M * N;
            launch_kernel(splitk_reduce_kernel, dim3((uint32_t)((total + kThreads - 1) / kThreads)), dim3(kThreads),
                               0, s, static_cast<const uint32_t *>(scratch), a.C, (uint32_t)splits, (uint32_t)(M * N),
                               total);
            be->pool.free(scratch, scratch_cls); // stream-ordered: later users queue behind the reduce
        }
#undef CG_MM_SWITCH
    } else {
        const uint64_t tiles = big ? tiles_big / batch : (uint64_t)((M + BM - 1) / BM) * ((N + 127) / 128);
        if (tiles > 0x7FFFFFFFull) return fail(CG_ERR_UNSUPPORTED, "matmul: too many tiles");
        dim3 grid((uint32_t)tiles, (uint32_t)batch);
        static const bool lds_ok = [] { // the tiles need more than the default 64 KiB of dynamic LDS
            bool ok = true;
#define CG_LDS(AF, BF)                                                                                                \
    ok &= hipFuncSetAttribute(reinterpret_cast<const void *>(&mfma_gemm_kernel<AF, BF, 4, 4, 1>),                     \
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)gemm_lds_bytes(256, 256, true)) == hipSuccess; \
    ok &= hipFuncSetAttribute(reinterpret_cast<const void *>(&mfma_gemm_kernel<AF, BF, 4, 4, 2>),                     \
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)gemm_lds_bytes(256, 256, true)) == hipSuccess;
            CG_LDS(true, true) CG_LDS(true, false) CG_LDS(false, true) CG_LDS(false, false)
#undef CG_LDS
            ok &= hipFuncSetAttribute(reinterpret_cast<const void *>(&mfma_gemm_kernel<false, false, 4, 4, 3>),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)gemm_lds_bytes(256, 256)) == hipSuccess;
            ok &= hipFuncSetAttribute(reinterpret_cast<const void *>(&mfma_gemm_kernel<false, false, 4, 4, 4>),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)gemm_lds_bytes(256, 256)) == hipSuccess;
            ok &= hipFuncSetAttribute(reinterpret_cast<const void *>(&mfma_gemm_kernel<false, false, 4, 4, 5>),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)gemm_lds_bytes(256, 256)) == hipSuccess;
            return ok;
        }();
        if (!lds_ok) return fail(CG_ERR_DEVICE, "matmul: cannot reserve %zu bytes of LDS", gemm_lds_bytes(128));
        if (big_packed) {
            const void *pa = x_native ? native_ptr(x) : nullptr, *pb = y_native ? native_ptr(y) : nullptr;
            void *ta = nullptr, *tb = nullptr;
            size_t ca = 0, cb = 0;
            // (the left operand's narrow copy is kept with its buffer when somebody else holds the activations too — q / k / v
            // and gate / up multiply the same ones —; an operand only this product reads is narrowed for it alone)
            const bool x_shared = x->rc.load() > 1 || x->buf->rc.load() > 1;
            int prc = x_native ? CG_OK : pack_operand(be, words_buffer(x), a.A, a.a_sm, a.a_sk, M, K, kind, x_shared, &pa, &ta, &ca);
            if (!prc && !y_native) prc = pack_operand(be, words_buffer(y), a.B, a.b_sn, a.b_sk, N, K, kind, true, &pb, &tb, &cb);
            if (prc) {
                (void)hipGetLastError();
                prc = kDeclined;
            } else {
                MmArgs p = a;
                p.A = static_cast<const uint32_t *>(pa);
                p.B = static_cast<const uint32_t *>(pb);
                p.K = (uint32_t)kw;
                p.a_sm = a_pitch;
                p.b_sn = b_pitch;
                p.a_sk = p.b_sk = 1;
                p.a_vec = p.b_vec = 1;
                p.c_fmt = (uint32_t)c_fmt;
                static const bool dlds_ok = [] {
                    bool ok = true;
#define CG_DLDS_LDS(H, NARROW)                                                                                                 \
    ok &= hipFuncSetAttribute(reinterpret_cast<const void *>(&mfma_gemm_dlds_kernel<H, NARROW>), hipFuncAttributeMaxDynamicSharedMemorySize, \
                              (int)kDldsLdsBytes) == hipSuccess;
                    CG_DLDS_LDS(3, false) CG_DLDS_LDS(3, true) CG_DLDS_LDS(4, false) CG_DLDS_LDS(4, true) CG_DLDS_LDS(5, false) CG_DLDS_LDS(5, true)
#undef CG_DLDS_LDS
                    return ok;
                }();
                if (dlds && !dlds_ok) prc = fail(CG_ERR_DEVICE, "matmul: cannot reserve %zu bytes of LDS", kDldsLdsBytes);
                else if (dlds) {
                    const bool narrow_out = c_fmt != kFmtWords;
                    const int64_t rest = N - wide_columns(be->compute_units, kind, M, N);
                    if (rest > 0) {
                        const int64_t first = N - rest;
                        const int trc = launch_narrow_tiles(be, kind, pa, a_pitch * per, M, static_cast<const uint32_t *>(pb) + first * b_pitch, b_pitch * per, rest, K,
                                                            static_cast<char *>(static_cast<void *>(a.C)) + first * (int64_t)fmt_bytes(c_fmt), c_fmt, N);
                        if (trc == CG_OK) p.n_tiles = (uint32_t)(first / 256);
                        else if (trc != kDeclined) prc = trc; // (declined: all of the columns below)
                    }
                    const uint64_t walked = p.n_tiles ? (uint64_t)p.n_tiles * ((M + 255) / 256) : tiles;
                    const dim3 pgrid((uint32_t)std::min<uint64_t>(walked, (uint64_t)be->compute_units)); // its workgroups walk the tiles
                    if (prc) {
                    } else
                    if (kind == 1 && narrow_out) launch_kernel((mfma_gemm_dlds_kernel<3, true>), pgrid, dim3(kThreads), kDldsLdsBytes, s, p);
                    else if (kind == 1) launch_kernel((mfma_gemm_dlds_kernel<3, false>), pgrid, dim3(kThreads), kDldsLdsBytes, s, p);
                    else if (kind == 2 && narrow_out) launch_kernel((mfma_gemm_dlds_kernel<4, true>), pgrid, dim3(kThreads), kDldsLdsBytes, s, p);
                    else if (kind == 2) launch_kernel((mfma_gemm_dlds_kernel<4, false>), pgrid, dim3(kThreads), kDldsLdsBytes, s, p);
                    else if (narrow_out) launch_kernel((mfma_gemm_dlds_kernel<5, true>), pgrid, dim3(kThreads), kDldsLdsBytes, s, p);
                    else launch_kernel((mfma_gemm_dlds_kernel<5, false>), pgrid, dim3(kThreads), kDldsLdsBytes, s, p);
                } else if (kind == 1) launch_kernel((mfma_gemm_kernel<false, false, 4, 4, 3>), grid, dim3(kThreads), gemm_lds_bytes(256, 256), s, p);
                else if (kind == 2) launch_kernel((mfma_gemm_kernel<false, false, 4, 4, 4>), grid, dim3(kThreads), gemm_lds_bytes(256, 256), s, p);
                else launch_kernel((mfma_gemm_kernel<false, false, 4, 4, 5>), grid, dim3(kThreads), gemm_lds_bytes(256, 256), s, p);
            }
            if (ta) be->pool.free(ta, ca); // stream-ordered: later users queue behind the product
            if (tb) be->pool.free(tb, cb);
            if (prc) return prc;
            hipError_t pe = hipGetLastError();
            return pe == hipSuccess ? CG_OK : hip_fail(pe, "matmul launch");
        }
#define CG_GEMM_HALF(AF, BF, H)                                                                                    \
    do {                                                                                                           \
        if (big)                                                                                                   \
            launch_kernel((mfma_gemm_kernel<AF, BF, 4, 4, H>), grid, dim3(kThreads), gemm_lds_bytes(256, 256, true), s, a); \
        else                                                                                                       \
            launch_kernel((mfma_gemm_kernel<AF, BF, 2, 2, H>), grid, dim3(kThreads), gemm_lds_bytes(128, 128, true), s, a); \
    } while (0)
#define CG_GEMM(AF, BF)                    \
    do {                                   \
        if (half == 2) CG_GEMM_HALF(AF, BF, 2); \
        else CG_GEMM_HALF(AF, BF, 1);      \
    } while (0)
        if (a_mfast) {
            if (b_nfast) CG_GEMM(true, true);
            else CG_GEMM(true, false);
        } else {
            if (b_nfast) CG_GEMM(false, true);
            else CG_GEMM(false, false);
        }
#undef CG_GEMM
#undef CG_GEMM_HALF
    }
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? CG_OK : hip_fail(e, "matmul launch");
}

int launch_matmul(cg_backend *be, const cg_tensor *x, const cg_tensor *y, cg_tensor *out, bool wide_only) {
    const int rc = product(be, x, y, out, wide_only, true);
    // no room to pack an operand: from words, as they lie or widened (a result in patterns is the caller's to ask for again in words)
    return rc == kDeclined && out && out->buf->fmt == kFmtWords ? product(be, x, y, out, wide_only, false) : rc;
}

} // namespace cg
