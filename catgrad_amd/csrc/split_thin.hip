// C[b, M, N] = A[b, M, K] B[b, K, N] of 32-bit floats for a few dozen rows, k contiguous in both operands, in pieces of bfloat16
// (split_tile.hpp: the same six piece products, the same scaling, the same sums without a direction).
#include "gemm_args.hpp"
#include "split_tile.hpp"

#include <algorithm>
#include <cmath>

namespace cg {
namespace {

using namespace split;
constexpr int kWaves = 8, kTurn = 32; // waves of a workgroup; values of k that a wave takes at a time

// 16 RT x 16 results per workgroup.  Its waves take turns of 32 values of k: a lane's 8 values of a row (32 of the 128 bytes that
// four lanes read) go from memory into the matrix instruction's registers as they lie, without LDS, two turns in flight; the
// waves' sums meet in LDS, so that k is cut eight ways without a second launch.  WHOLE: k is whole turns.
//
// Such products are bound by latency: on 64 x 64 tiles a workgroup walks its stages one after the other, and a second launch adds
// the parts that k is cut into.  Both launches there, and here, in us: 64 x 512 x 256 9.2 and 4.2, 32 x 1536 x 576 11.9 and 5.8,
// 64 x 1024 x 1024 13.7 and 7.6, 32 x 3072 x 1024 15.2 and 9.5, 16 x 8192 x 2048 24.7 and 18.7.  A turn is 0.97 us for one row block
// and two waves per SIMD: 56 vector instructions split 8 values, twice, against six matrix instructions.  Measured and left out: four
// turns in flight (their loads are asked for again where there are fewer turns: 64 x 512 x 256 6.6), sixteen waves (up to 40 % more).
template <int RT, bool WHOLE> __global__ __launch_bounds__(64 * kWaves, 4) void split_thin_kernel(const MmArgs a) {
    constexpr uint32_t TILE = RT * 256;
    __shared__ float red[kWaves][TILE];
    __shared__ float2v tops[kWaves];
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64, li = lane % 16, lg = lane / 16;
    const uint32_t n0 = blockIdx.x * 16, m0 = blockIdx.y * (16 * RT), K = a.K, turns = (K + kTurn - 1) / kTurn;
    int64_t pa, pb;
    batch_offsets(a, blockIdx.z, pa, pb);
    const float *const A = reinterpret_cast<const float *>(a.A) + pa, *const B = reinterpret_cast<const float *>(a.B) + pb;
    const float *row[RT], *const col = B + (int64_t)min(n0 + li, a.N - 1) * a.b_sn;
#pragma unroll
    for (int i = 0; i < RT; i++) row[i] = A + (int64_t)min(m0 + 16 * i + li, a.M - 1) * a.a_sm; // (rows behind the last repeat it)
    float4v x[2][RT][2], y[2][2];
    auto ask = [&](const uint32_t t, const int set) {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const uint32_t k0 = t * kTurn + lg * 8 + h * 4, k = WHOLE ? k0 : min(k0, K - 4);
            y[set][h] = *reinterpret_cast<const float4v *>(col + k);
#pragma unroll
            for (int i = 0; i < RT; i++) x[set][i][h] = *reinterpret_cast<const float4v *>(row[i] + k);
        }
    };
    // (values behind the last, which were read elsewhere, become zeros)
    auto there = [&](const uint32_t t, const int h, const float4v v) {
        const bool in = WHOLE || t * kTurn + lg * 8 + h * 4 < K;
        float4v r;
#pragma unroll
        for (int j = 0; j < 4; j++) r[j] = in ? v[j] : 0.0f;
        return r;
    };
    float4v acc[RT];
    const float4v zero = {};
#pragma unroll
    for (int i = 0; i < RT; i++) acc[i] = zero;
    float ta = 0.0f, tb = 0.0f; // largest magnitudes
    auto pieces = [&](const float4v u, const float4v v, const float up, float &top, bf16x8 (&p)[3]) {
        uint32_t w[4][3];
        split2(u[0] * up, u[1] * up, w[0]);
        split2(u[2] * up, u[3] * up, w[1]);
        split2(v[0] * up, v[1] * up, w[2]);
        split2(v[2] * up, v[3] * up, w[3]);
        grow(top, u[0], u[1]);
        grow(top, u[2], u[3]);
        grow(top, v[0], v[1]);
        grow(top, v[2], v[3]);
#pragma unroll
        for (int q = 0; q < 3; q++) {
            const uint4 z = make_uint4(w[0][q], w[1][q], w[2][q], w[3][q]);
            p[q] = __builtin_bit_cast(bf16x8, z);
        }
    };
    auto multiply = [&](const uint32_t t, const int set, const bool turned) { // (turned: of the negated left operand, taken away)
        const float up = turned ? -kUp : kUp, down = turned ? -kDown : kDown;
        bf16x8 p[3], q[3];
        pieces(there(t, 0, y[set][0]), there(t, 1, y[set][1]), kUp, tb, q);
#pragma unroll
        for (int i = 0; i < RT; i++) {
            pieces(there(t, 0, x[set][i][0]), there(t, 1, x[set][i][1]), up, ta, p);
            float4v sum = zero;
#pragma unroll
            for (int g = 0; g < 6; g++) sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(p[kPairA[g]], q[kPairB[g]], sum, 0, 0, 0);
#pragma unroll
            for (int v = 0; v < 4; v++) acc[i][v] = __builtin_fmaf(sum[v], down, acc[i][v]);
            // (Kept in front of the branch behind a turn: sunk into both of its sides, the sums were read before the matrix
            // instruction had written them, whose wait the compiler does not place there.)
            asm volatile("" : "+v"(acc[i]));
        }
    };
    if (wave < turns) { // (the loads stay where they stand, and every wait in the loop knows what else is on its way)
        const uint32_t n = (turns - 1 - wave) / kWaves + 1;
        const bool odd = wave % 2;
        uint32_t t = wave;
        ask(t, 0);
        if (n == 1) {
            multiply(t, 0, odd);
        } else {
            ask(t + kWaves, 1);
            for (uint32_t left = n; left > 3; left -= 2, t += 2 * kWaves) {
                multiply(t, 0, odd);
                __builtin_amdgcn_sched_barrier(0);
                ask(t + 2 * kWaves, 0);
                __builtin_amdgcn_sched_barrier(0);
                multiply(t + kWaves, 1, !odd);
                __builtin_amdgcn_sched_barrier(0);
                ask(t + 3 * kWaves, 1);
                __builtin_amdgcn_sched_barrier(0);
            }
            multiply(t, 0, odd);
            if (n % 2) {
                ask(t + 2 * kWaves, 0);
                multiply(t + kWaves, 1, !odd);
                multiply(t + 2 * kWaves, 0, odd);
            } else {
                multiply(t + kWaves, 1, !odd);
            }
        }
    }
    auto leave = [&]() {
#pragma unroll
        for (int i = 0; i < RT; i++)
#pragma unroll
            for (int v = 0; v < 4; v++) red[wave][i * 256 + v * 64 + lane] = acc[i][v];
    };
    leave();
    const float2v top = {wave_max(ta), wave_max(tb)};
    if (lane == 0) tops[wave] = top;
    __syncthreads();
    float2v most = tops[0];
#pragma unroll
    for (int w = 1; w < kWaves; w++) most = {fmaxf(most[0], tops[w][0]), fmaxf(most[1], tops[w][1])};
    if (!__builtin_amdgcn_readfirstlane(in_range(most[0], most[1]))) { // the 32-bit instructions, for what the pieces do not hold
        __syncthreads();
#pragma unroll
        for (int i = 0; i < RT; i++) acc[i] = zero;
        for (uint32_t t = wave; t < turns; t += kWaves) {
            ask(t, 0);
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const float4v w = there(t, h, y[0][h]);
#pragma unroll
                for (int i = 0; i < RT; i++) {
                    const float4v u = there(t, h, x[0][i][h]);
#pragma unroll
                    for (int j = 0; j < 4; j++) acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(u[j], w[j], acc[i], 0, 0, 0);
                }
            }
        }
        leave();
        __syncthreads();
    }
    uint32_t *const C = a.C + ((uint64_t)blockIdx.z * a.M + m0) * a.N;
    for (uint32_t e = threadIdx.x; e < TILE; e += 64 * kWaves) {
        float s = red[0][e];
#pragma unroll
        for (int w = 1; w < kWaves; w++) s += red[w][e];
        const uint32_t l = e % 64, r = e / 256 * 16 + l / 16 * 4 + e / 64 % 4, c = n0 + l % 16;
        if (m0 + r < a.M && c < a.N) C[(uint64_t)r * a.N + c] = asu(s);
    }
}

} // namespace

// What a launch takes, in microseconds: before and behind the turns, and eight waves' turns of a workgroup, times the workgroups that a
// compute unit takes.  Fitted to 176 shapes of 9 to 256 rows, 10 to 16000 columns and 64 to 8192 values of k, both heights timed:
// one row block up to a workgroup per compute unit, two beyond, where the columns' pieces are worth sharing (64 x 4096 x 1024 15.3
// against 19.4 us).  Four row blocks were within 7 % of the better of these and of the tiles where they were the fastest at all.
double thin_gemm_cost(const cg_backend *be, const MmArgs &a, int *high) {
    double best = 0;
    for (int rt = 1; rt <= 2; rt++) {
        const uint64_t rows = (a.M + 16 * rt - 1) / (16 * rt);
        if (rows > 65535 || a.batch > 65535) continue;
        const double rounds = (double)(rows * ((a.N + 15) / 16) * a.batch) / be->compute_units;
        const double us = 3.2 + (rt == 1 ? 0.97 : 1.43) * std::max(0.25, a.K / (8.0 * kTurn)) * std::max(1.0, rounds);
        if (best == 0 || us < best) best = us, *high = rt;
    }
    return best;
}

int launch_thin_gemm(cg_backend *be, const MmArgs &a, int high) {
    const dim3 grid((a.N + 15) / 16, (a.M + 16 * high - 1) / (16 * high), a.batch), block(64 * kWaves);
    if (a.K % kTurn == 0) {
        if (high == 1) launch_kernel((split_thin_kernel<1, true>), grid, block, 0, be->stream, a);
        else launch_kernel((split_thin_kernel<2, true>), grid, block, 0, be->stream, a);
    } else {
        if (high == 1) launch_kernel((split_thin_kernel<1, false>), grid, block, 0, be->stream, a);
        else launch_kernel((split_thin_kernel<2, false>), grid, block, 0, be->stream, a);
    }
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? CG_OK : hip_fail(e, "matmul launch");
}

} // namespace cg
