// Interpreter kernels for deferred element-wise expressions (see `Pending` in common.hpp).
//
// A program is a short list of instructions over a register file of 16 values per
// element: the leaves (strided views or immediates, loaded once) occupy the first
// registers, every instruction names its destination (allocated on the host).  Every lane runs the same program, so the
// register numbers and op codes are wave-uniform: the register file lives in VGPRs and is
// indexed with scalar (uniform) indices, and the op switch is a scalar branch.  Arithmetic
// is the same `apply<OP, F>` the single-op kernels use, applied in the same order, so a
// fused chain is bit-identical to the chain of separate kernels — it just reads every leaf
// once and writes once.
//
//   fused_kernel         value of the program -> dense or strided output      (HBM-bound:
//                        4 B per distinct leaf element + 4 B per output element)
//   fused_reduce_kernel  sum / max / argmax over the last axis of the value   (HBM-bound:
//                        4 B per distinct leaf element + 4 B per row)
#include "interp.hpp"

namespace cg {

bool fused_program_fits(const Pending &p) {
    uint8_t phys[kMaxLeaves + kMaxInstr];
    return allocate_registers(p, phys);
}

// ---- g / (1 + exp(-g)) * u of dense bfloat16 or fp8 tensors, rounded after every operation ------------------------------
// The bits of MapSiluMulBF16 / MapSiluMulF8, whose kernels are bound by the exponential and the division (8192 x 8192 bf16: 116 us =
// 3.5 TB/s; 1500 x 8192 fp8: 30 us = 1.2): what is left here is the memory's time, 16 bytes a lane and tensor: 79 us = 5.1 TB/s; 17.
//
// bf16, |g| <= 64 (everything else goes through the program's operations): exp(-g) is the hardware's 2^y with y's rounding and the
// low part of log2 e put back as a factor, which rounds to the same bfloat16 as the exact function for every such g (all of them are
// compared in the tests).  g / d is g times the hardware's reciprocal, off by less than 2^-22 of it: a quotient of two 8-bit
// significands lies at least 2^-17 of itself from the middle between two bfloat16 numbers, so it rounds as the exact one does
// (d, a rounded 1 + exp(-g), is between 1 and 2^93; subnormal g have d = 2 and an exact product).
//
// f16 stays with MapSiluMulF16: quotients of its 11-bit significands come as close to the middle as 2^-23 of themselves, nearer than the
// reciprocal is to them, so the same steps would not give its bits.
template <int R> __device__ __forceinline__ uint32_t silu_exact(uint32_t g, uint32_t one) {
    const uint32_t e = apply<R, true>(apply<kExp, true>(apply<kNeg, true>(g, 0, 0, nullptr), 0, 0, nullptr), 0, 0, nullptr);
    const uint32_t d = apply<R, true>(apply<kAdd, true>(one, e, 0, nullptr), 0, 0, nullptr);
    return apply<R, true>(apply<kDiv, true>(g, d, 0, nullptr), 0, 0, nullptr);
}
__device__ __forceinline__ uint32_t cvt_bf16_pair(float x, float y) {
    const float2cv v = {x, y};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2cv));
}
__global__ __launch_bounds__(kBlock) void silu_mul_bf16_kernel(const uint16_t *g, const uint16_t *u, uint16_t *y, uint64_t n) {
    constexpr uint32_t kOne = 0x3F800000u;
    const uint64_t at = ((uint64_t)blockIdx.x * kBlock + threadIdx.x) * 8;
    if (at >= n) return;
    if (at + 8 > n) { // the last few
        for (uint64_t i = at; i < n; i++) y[i] = (uint16_t)(round_bf16_bits(apply<kMul, true>(silu_exact<kRoundBF16>((uint32_t)g[i] << 16, kOne), (uint32_t)u[i] << 16, 0, nullptr)) >> 16);
        return;
    }
    const uint4 gq = *reinterpret_cast<const uint4 *>(g + at), uq = *reinterpret_cast<const uint4 *>(u + at);
    const uint32_t gw[4] = {gq.x, gq.y, gq.z, gq.w}, uw[4] = {uq.x, uq.y, uq.z, uq.w};
    uint32_t yw[4], most = 0; // (the largest magnitude's pattern)
#pragma unroll
    for (int i = 0; i < 4; i++) most = max(most, max(gw[i] & 0x7FFFu, (gw[i] >> 16) & 0x7FFFu));
    if (most <= 0x4280u) { // 64
        constexpr float kLog2e = 0x1.715476p+0f, kLog2eLow = 0x1.4ae0cp-26f, kLn2 = 0x1.62e43p-1f;
        auto exp_neg = [&](float x) {
            const float t = x * -kLog2e, rest = __builtin_fmaf(x, -kLog2eLow, __builtin_fmaf(x, -kLog2e, -t));
            const float e = __builtin_amdgcn_exp2f(t);
            return __builtin_fmaf(e, rest * kLn2, e);
        };
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float g0 = asf(gw[i] << 16), g1 = asf(gw[i] & 0xFFFF0000u);
            const uint32_t e = cvt_bf16_pair(exp_neg(g0), exp_neg(g1));
            const uint32_t d = cvt_bf16_pair(1.0f + asf(e << 16), 1.0f + asf(e & 0xFFFF0000u));
            const uint32_t s = cvt_bf16_pair(g0 * __builtin_amdgcn_rcpf(asf(d << 16)), g1 * __builtin_amdgcn_rcpf(asf(d & 0xFFFF0000u)));
            yw[i] = cvt_bf16_pair(asf(s << 16) * asf(uw[i] << 16), asf(s & 0xFFFF0000u) * asf(uw[i] & 0xFFFF0000u));
        }
    } else {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t lo = apply<kMul, true>(silu_exact<kRoundBF16>(gw[i] << 16, kOne), uw[i] << 16, 0, nullptr);
            const uint32_t hi = apply<kMul, true>(silu_exact<kRoundBF16>(gw[i] & 0xFFFF0000u, kOne), uw[i] & 0xFFFF0000u, 0, nullptr);
            yw[i] = round_bf16_bits(lo) >> 16 | round_bf16_bits(hi);
        }
    }
    *reinterpret_cast<uint4 *>(y + at) = make_uint4(yw[0], yw[1], yw[2], yw[3]);
}
// fp8: the 256 values of g / (1 + exp(-g)) from the program's operations, a thread each, then 64 values of the tensors per thread
constexpr uint32_t kSiluTrips = 4;
__global__ __launch_bounds__(kBlock) void silu_mul_f8_kernel(const uint8_t *g, const uint8_t *u, uint8_t *y, uint64_t n, uint32_t one) {
    static_assert(kBlock == 256, "a thread per pattern");
    __shared__ uint32_t silu[256];
    silu[threadIdx.x] = silu_exact<kRoundF8>(f8_word_of((uint8_t)threadIdx.x), one);
    __syncthreads();
    auto value = [&](uint32_t gb, uint32_t ub) { return (uint32_t)f8_byte_of(round_f8_bits(apply<kMul, true>(silu[gb], f8_word_of((uint8_t)ub), 0, nullptr))); };
#pragma unroll
    for (uint32_t t = 0; t < kSiluTrips; t++) {
        const uint64_t at = (((uint64_t)blockIdx.x * kSiluTrips + t) * kBlock + threadIdx.x) * 16;
        if (at >= n) return;
        if (at + 16 > n) {
            for (uint64_t i = at; i < n; i++) y[i] = (uint8_t)value(g[i], u[i]);
            return;
        }
        const uint4 gq = *reinterpret_cast<const uint4 *>(g + at), uq = *reinterpret_cast<const uint4 *>(u + at);
        const uint32_t gw[4] = {gq.x, gq.y, gq.z, gq.w}, uw[4] = {uq.x, uq.y, uq.z, uq.w};
        uint32_t yw[4] = {};
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int b = 0; b < 4; b++) yw[i] |= value(gw[i] >> (8 * b) & 0xFFu, uw[i] >> (8 * b) & 0xFFu) << (8 * b);
        *reinterpret_cast<uint4 *>(y + at) = make_uint4(yw[0], yw[1], yw[2], yw[3]);
    }
}
// Both tensors and the result dense in one of the two formats, from 16-byte addresses; bf16: the constant is one.
static bool launch_dense_silu_mul(const Pending &p, const FusedArgs &a, LaunchQueue &s) {
    const bool bf16 = program_matches<MapSiluMulBF16>(p);
    if (!bf16 && !program_matches<MapSiluMulF8>(p)) return false;
    const uint32_t fmt = bf16 ? kFmtBF16 : kFmtF8;
    auto dense = [&](const Operand &o) { return o.fmt == fmt && o.is == 1 && !o.uniform && reinterpret_cast<uintptr_t>(o.ptr) % 16 == 0; };
    if (a.g.nouter != 0 || !dense(a.leaf[0]) || !dense(a.leaf[2]) || !dense(a.out)) return false;
    if (bf16 && a.leaf[1].ubits != 0x3F800000u) return false;
    const uint64_t n = a.g.inner, per = bf16 ? kBlock * 8 : kBlock * 16 * kSiluTrips;
    const dim3 grid((uint32_t)((n + per - 1) / per));
    if (bf16)
        launch_kernel(silu_mul_bf16_kernel, grid, dim3(kBlock), 0, s, reinterpret_cast<const uint16_t *>(a.leaf[0].ptr),
                           reinterpret_cast<const uint16_t *>(a.leaf[2].ptr), reinterpret_cast<uint16_t *>(const_cast<char *>(a.out.ptr)), n);
    else
        launch_kernel(silu_mul_f8_kernel, grid, dim3(kBlock), 0, s, reinterpret_cast<const uint8_t *>(a.leaf[0].ptr),
                           reinterpret_cast<const uint8_t *>(a.leaf[2].ptr), reinterpret_cast<uint8_t *>(const_cast<char *>(a.out.ptr)), n, a.leaf[1].ubits);
    return true;
}

int launch_fused(cg_backend *be, const cg_tensor *out, const Pending &p) {
    if (int frc = flush_deferred(be)) return frc;
    FusedArgs a;
    double bytes;
    bool full;
    int rc = fill_args(be, p, out->dims, out->rank, out, false, &a, &bytes, &full);
    if (rc) return rc;
    if (a.g.total == 0) return CG_OK;
    trace_program(be, p, p.ninstr, "map", out->dims, out->rank);
    ProfScope prof(be, CG_K_ELEMENTWISE, bytes + distinct_bytes(out));
    dim3 grid((uint32_t)((a.g.total + kBlock - 1) / kBlock)), block(kBlock);
    if (be->aot && (launch_dense_silu_mul(p, a, be->stream) || aot_map_dispatch(p, a, grid, be->stream, MapPrograms{}))) {
        be->programs_compiled++;
        hipError_t e = hipGetLastError();
        return e == hipSuccess ? CG_OK : hip_fail(e, "compiled element-wise launch");
    }
    be->programs_interpreted++;
    if (a.g.vec == 4) {
        if (full)
            launch_kernel((fused_kernel<4, true>), grid, block, 0, be->stream, a);
        else
            launch_kernel((fused_kernel<4, false>), grid, block, 0, be->stream, a);
    } else {
        if (full)
            launch_kernel((fused_kernel<1, true>), grid, block, 0, be->stream, a);
        else
            launch_kernel((fused_kernel<1, false>), grid, block, 0, be->stream, a);
    }
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? CG_OK : hip_fail(e, "fused element-wise launch");
}

// Two or three element-wise results in one launch; declines unless every program is one the
// grouped kernel holds (rotary embedding, strided copy).
int launch_fused_group(cg_backend *be, const cg_tensor *const *outs, const Pending *const *ps, int n) {
    if (!be->aot || n < 2 || n > kMaxMapGroup) return kDeclined;
    FusedGroup g;
    double bytes = 0;
    uint32_t blocks = 0;
    for (int i = 0; i < n; i++) {
        const Pending &p = *ps[i];
        if (program_matches<MapRope>(p))
            g.prog[i] = 0;
        else if (p.nleaf == 1 && p.ninstr == 1 && p.nred == 0 && (p.ins[0].op & ~kInstrU32) == kCopy && p.ins[0].a == 0 &&
                 !p.leaf[0].uniform && !p.leaf[0].pw)
            g.prog[i] = 1;
        else
            return kDeclined;
        double b;
        bool full;
        int rc = fill_args(be, p, outs[i]->dims, outs[i]->rank, outs[i], false, &g.p[i], &b, &full);
        if (rc) return rc;
        if (g.p[i].g.total == 0) return kDeclined;
        bytes += b + distinct_bytes(outs[i]);
        g.first[i] = blocks;
        blocks += (uint32_t)((g.p[i].g.total + kBlock - 1) / kBlock);
    }
    g.first[n] = blocks;
    g.n = (uint32_t)n;
    for (int i = 0; i < n; i++) trace_program(be, *ps[i], ps[i]->ninstr, "map (grouped)", outs[i]->dims, outs[i]->rank);
    ProfScope prof(be, CG_K_ELEMENTWISE, bytes);
    launch_kernel(aot_map_group_kernel, dim3(blocks), dim3(kBlock), 0, be->stream, g);
    be->programs_compiled += n;
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? CG_OK : hip_fail(e, "grouped element-wise launch");
}

int launch_fused_reduce(cg_backend *be, int kind, bool f32, const Pending &p, int ninstr, const int64_t *dims, int rank,
                        cg_tensor *out) {
    if (int frc = flush_deferred(be)) return frc;
    FusedArgs a;
    double bytes;
    bool full;
    int rc = fill_args(be, p, dims, rank, nullptr, true, &a, &bytes, &full, ninstr);
    if (rc) return rc;
    a.n = a.g.inner;
    uint64_t rows = 1;
    for (uint32_t d = 0; d < a.g.nouter; d++) rows *= a.g.od[d];
    if (rows > 0xFFFFFFFFull) return fail(CG_ERR_UNSUPPORTED, "reduction extents above 2^32-1");
    a.rows = (uint32_t)rows;
    uint32_t *op = static_cast<uint32_t *>(out->buf->ptr);
    be->programs_interpreted++;
    trace_program(be, p, ninstr, kind == kSum ? "reduce-sum" : kind == kMax ? "reduce-max" : "reduce-argmax", dims, rank);
    ProfScope prof(be, CG_K_REDUCE, bytes + distinct_bytes(out));
    uint32_t want = (a.n + 7) / 8;
    int tpr = want <= 4 ? 4 : want <= 16 ? 16 : want <= 64 ? 64 : 256;
    uint32_t rpb = kBlock / tpr;
    dim3 grid((a.rows + rpb - 1) / rpb), block(kBlock);
    const int f = f32 ? 1 : 0;
#define CG_LAUNCH(VEC, TPR)                                                                                  \
    do {                                                                                                     \
        if (full)                                                                                            \
            launch_kernel((fused_reduce_kernel<VEC, TPR, true>), grid, block, 0, be->stream, a, op, kind, f);  \
        else                                                                                                 \
            launch_kernel((fused_reduce_kernel<VEC, TPR, false>), grid, block, 0, be->stream, a, op, kind, f); \
    } while (0)
    if (a.g.vec == 4) {
        switch (tpr) {
        case 4: CG_LAUNCH(4, 4); break;
        case 16: CG_LAUNCH(4, 16); break;
        case 64: CG_LAUNCH(4, 64); break;
        default: CG_LAUNCH(4, 256); break;
        }
    } else {
        switch (tpr) {
        case 4: CG_LAUNCH(1, 4); break;
        case 16: CG_LAUNCH(1, 16); break;
        case 64: CG_LAUNCH(1, 64); break;
        default: CG_LAUNCH(1, 256); break;
        }
    }
#undef CG_LAUNCH
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? CG_OK : hip_fail(e, "fused reduction launch");
}

} // namespace cg
